// Shared by the kernels for 16-bit tensors that keep their LDS images in the tensors' own format (two elements
// per dword): the image layout, how it is filled, and the two-element dot product.
#pragma once

#include "dwconv_tile_common.hpp"

namespace dwconv {

constexpr int kPadL = 8;  // element j of an image row holds input column j - kPadL

// `planes` images of `lds_rows` rows of `pitch` 16-bit elements; a row is written in slots of eight elements
// (four dwords), `spr` of them, the first of which lies wholly left of the plane.
// In LDS a slot takes FIVE dwords, the fifth unused: lanes that own consecutive 8-element blocks then sit five
// dwords apart, an odd stride, and their two-dword reads fall on distinct banks.  With the slots packed (stride
// four) the same reads use half the banks twice over: the counters showed the LDS busy 60 % of the time, two thirds
// of it in bank conflicts.
struct Image16 {
    int in_h, in_w, in_plane;   // in_w is a multiple of eight, unless the rows are staged with ANY
    int lds_rows;
    unsigned lds_rows_magic;
    int spr;
    unsigned spr_magic;
    int pitch;                  // elements per image row, a multiple of eight
    int rp;                     // dwords per image row in LDS: five per slot
    int pp;                     // dwords per plane image in LDS
};

// Row pitch and slots for windows that reach input column `last_col` at most.
inline void layout_image16(Image16 &im, int last_col)
{
    im.spr = ceil_div(kPadL + std::max(last_col + 1, im.in_w), 8);
    // eight spare elements per row keep the rows of consecutive row blocks off the same banks
    im.pitch = 8 * im.spr + 8;
    im.rp = 5 * (im.pitch / 8);
}

// False if the 16-bit reciprocals or the 24-bit multiplies of stage_image16 would not be exact.
inline bool finish_image16(Image16 &im, int lds_rows, int planes_per_tile)
{
    im.lds_rows = lds_rows;
    im.pp = lds_rows * im.rp;
    if (static_cast<long>(planes_per_tile) * lds_rows * im.spr >= 65536) return false;
    if (im.in_h >= (1 << 23) || im.in_w >= (1 << 23) || (planes_per_tile > 1 && im.in_plane >= (1 << 23))) return false;
    if (static_cast<long>(planes_per_tile) * im.in_plane * 2 >= static_cast<long>(kOob)) return false;
    im.spr_magic = magic_u16(im.spr);
    im.lds_rows_magic = magic_u16(lds_rows);
    return true;
}

// LDS dword of logical dword j of an image row (four data dwords per five).
__host__ __device__ constexpr int swz(int j) { return j + (j >> 2); }

template <typename IO>
__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c)
{
    if constexpr (std::is_same<IO, bf16_t>::value) {
        typedef __bf16 v2 __attribute__((ext_vector_type(2)));
        return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2, a), __builtin_bit_cast(v2, b), c, false);
    } else {
        typedef _Float16 v2 __attribute__((ext_vector_type(2)));
        return __builtin_amdgcn_fdot2(__builtin_bit_cast(v2, a), __builtin_bit_cast(v2, b), c, false);
    }
}

// Fills the images of `nplanes` planes starting at `src` (plane stride im.in_plane) with input rows iy0 ...: every
// slot of every row is written, with zeros (loads beyond the view) outside the plane.  `image` is the first dword,
// `dump` the index of a spare slot.  A lane keeps its column and walks down the rows: per slot two additions, a range check and a
// select.  kBatch loads are in flight per lane.
// ANY: rows of any width that start on any element.  A slot's load starts on a 32-bit boundary: 128 bits at a multiple of 4
// where every row does; where some start 2 bytes past one, a fifth dword and four funnel shifts when the slot enters LDS.
// What a row's last slot read of the next row is masked there too (the masks belong to the lane's column).
template <typename IO, int kBatch = 4, bool ANY = false>
__device__ __forceinline__ void stage_image16(const Image16 &im, const IO *src, uint32_t *image, int dump, int nplanes, int iy0)
{
    const bool split = ANY && mixed_row_starts(src, im.in_w);
    AnyWidthView wide{};
    if constexpr (ANY) wide = any_width_view(src, static_cast<long>(nplanes) * im.in_plane * sizeof(IO));
    else wide.view = buffer_view(src, static_cast<long>(nplanes) * im.in_plane * sizeof(IO));
    struct Slot {
        u32x4 v;
        unsigned more, shift;  // split rows: the dword behind v, and how far the slot starts inside its first dword
    };
    auto load = [&](unsigned off) {
        Slot s;
        if (ANY && split) {
            const unsigned at = off < kOob ? off + wide.bias : kOob;
            s.v = __builtin_amdgcn_raw_buffer_load_b128(wide.view, at & ~3u, 0, 0);
            s.more = __builtin_amdgcn_raw_buffer_load_b32(wide.view, (at & ~3u) + 16u, 0, 0);
            s.shift = (at & 2u) << 3;
        } else {
            s.v = __builtin_amdgcn_raw_buffer_load_b128(wide.view, off, 0, 0);
            s.more = s.shift = 0u;
        }
        return s;
    };
    const int nthreads = blockDim.x;
    const int rpp_raw = fast_div(nthreads, im.spr_magic);
    const int rpp = max(rpp_raw, 1);                     // rows per pass of the workgroup
    const int col_step = rpp_raw ? im.spr : nthreads;    // one trip unless a row has more slots than lanes
    const int rl = fast_div(threadIdx.x, im.spr_magic);
    const int spitch = im.pitch >> 3;                    // in slots
    u32x4 keep = {~0u, ~0u, ~0u, ~0u};  // ANY: the elements of the lane's column that belong to its rows
    auto put = [&](int slot, const Slot &s) {
        u32x4 v = s.v;
        if constexpr (ANY) {
            if (split) {
                v.x = __builtin_amdgcn_alignbit(s.v.y, s.v.x, s.shift);
                v.y = __builtin_amdgcn_alignbit(s.v.z, s.v.y, s.shift);
                v.z = __builtin_amdgcn_alignbit(s.v.w, s.v.z, s.shift);
                v.w = __builtin_amdgcn_alignbit(s.more, s.v.w, s.shift);
            }
            v &= keep;
        }
        uint32_t *d = image + slot * 5;
        d[0] = v.x;
        d[1] = v.y;
        d[2] = v.z;
        d[3] = v.w;
    };
    if (rl >= rpp) return;
    for (int sc = threadIdx.x - __mul24(rl, im.spr); sc < im.spr; sc += col_step) {
        const int ix = 8 * sc - kPadL;
        const bool col_ok = static_cast<unsigned>(ix) < static_cast<unsigned>(im.in_w);
        if constexpr (ANY) {
            const int n = im.in_w - ix;  // elements of the row from this column on
#pragma unroll
            for (int d = 0; d < 4; ++d) keep[d] = n > 2 * d + 1 ? ~0u : (n > 2 * d ? 0xffffu : 0u);
        }
        if (nplanes == 1) {
            const int lo = max(iy0, 0);
            const unsigned span = static_cast<unsigned>(max(min(im.in_h, iy0 + im.lds_rows) - lo, 0));
            const unsigned off_step = __mul24(rpp, im.in_w) * 2u;
            const int dst_step = __mul24(rpp, spitch);
            int iy = iy0 + rl;
            unsigned off = (__mul24(iy, im.in_w) + ix) * 2u;
            int dst = __mul24(rl, spitch) + sc;
            int rb = 0;
            // whole batches (uniform bound, unconditional stores), then one batch whose rows past the image go to
            // the spare slot.  A store under a per-lane condition would drag its load into the conditional block,
            // behind the other loads' wait.
            for (; rb + rpp * kBatch <= im.lds_rows; rb += rpp * kBatch) {
                Slot v[kBatch];
#pragma unroll
                for (int u = 0; u < kBatch; ++u) {
                    const bool ok = col_ok && static_cast<unsigned>(iy + u * rpp - lo) < span;
                    v[u] = load(ok ? off + u * off_step : kOob);
                }
#pragma unroll
                for (int u = 0; u < kBatch; ++u) put(dst + u * dst_step, v[u]);
                iy += rpp * kBatch;
                off += off_step * kBatch;
                dst += dst_step * kBatch;
            }
            if (rb < im.lds_rows) {
                Slot v[kBatch];
#pragma unroll
                for (int u = 0; u < kBatch; ++u) {
                    const bool ok = col_ok && static_cast<unsigned>(iy + u * rpp - lo) < span;
                    v[u] = load(ok ? off + u * off_step : kOob);
                }
#pragma unroll
                for (int u = 0; u < kBatch; ++u) put(rb + rl + u * rpp < im.lds_rows ? dst + u * dst_step : dump, v[u]);
            }
        } else {
            const int total_rows = nplanes * im.lds_rows;
            const int pslots = im.lds_rows * spitch;
            for (int ra = rl; ra < total_rows; ra += rpp * kBatch) {
                Slot v[kBatch];
                int dst[kBatch];
#pragma unroll
                for (int u = 0; u < kBatch; ++u) {
                    const bool live = ra + u * rpp < total_rows;
                    const int rc = min(ra + u * rpp, total_rows - 1);
                    const int pl = fast_div(rc, im.lds_rows_magic);
                    const int r = rc - __mul24(pl, im.lds_rows);
                    const int iy = iy0 + r;
                    const bool ok = live && col_ok && static_cast<unsigned>(iy) < static_cast<unsigned>(im.in_h);
                    const unsigned off = (__mul24(pl, im.in_plane) + __mul24(iy, im.in_w) + ix) * 2u;
                    v[u] = load(ok ? off : kOob);
                    dst[u] = live ? __mul24(pl, pslots) + __mul24(r, spitch) + sc : dump;
                }
#pragma unroll
                for (int u = 0; u < kBatch; ++u) put(dst[u], v[u]);
            }
        }
    }
}

// `n` packed results (n <= 2 NP) into a run of consecutive 16-bit elements in LDS, from element `at` on, which need not be
// even.  A whole group goes as NP - 1 dwords on 32-bit boundaries and the two elements that are left: the first two where the
// group starts on such a boundary, the first and the last where it does not.
template <int NP>
__device__ __forceinline__ void lds_put_run16(uint16_t *run, int at, int n, const uint32_t (&v)[NP])
{
    uint16_t *d = run + at;
    if (n >= 2 * NP) {
        const bool odd = (at & 1) != 0;
        uint32_t *mid = reinterpret_cast<uint32_t *>(d + (odd ? 1 : 2));
#pragma unroll
        for (int i = 0; i + 1 < NP; ++i) mid[i] = odd ? __builtin_amdgcn_alignbit(v[i + 1], v[i], 16) : v[i + 1];
        d[0] = static_cast<uint16_t>(v[0]);
        d[odd ? 2 * NP - 1 : 1] = static_cast<uint16_t>((odd ? v[NP - 1] : v[0]) >> 16);
    } else {
#pragma unroll
        for (int e = 0; e < 2 * NP - 1; ++e)
            if (e < n) d[e] = static_cast<uint16_t>(v[e / 2] >> (16 * (e & 1)));
    }
}
// A run of 16-bit results that starts on any element: lds[head .. head + n) leaves for to[0 .. n), `head` being the elements
// between the 16-byte boundary before `to` and `to` (run_head).  Whole 16-byte pieces leave as such, the two ends element by
// element.  The workgroup calls it together, after a barrier behind the writes into LDS.
template <typename IO>
__device__ __forceinline__ void store_run16(IO *to, const uint16_t *lds, int head, int n)
{
    uint16_t *const base = reinterpret_cast<uint16_t *>(to) - head;
    const int end = head + n;
    const __amdgpu_buffer_rsrc_t view = buffer_view(base, static_cast<long>(end) * 2);
    for (int c = threadIdx.x * 8; c < end; c += blockDim.x * 8) {
        if (c >= head && c + 8 <= end) {
            __builtin_amdgcn_raw_buffer_store_b128(*reinterpret_cast<const u32x4 *>(lds + c), view, c * 2u, 0, kStoreStreaming);
        } else {
            for (int e = max(c, head); e < min(c + 8, end); ++e) base[e] = lds[e];
        }
    }
}

}  // namespace dwconv
