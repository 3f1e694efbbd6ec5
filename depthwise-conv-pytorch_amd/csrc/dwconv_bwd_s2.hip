// Fused backward pass (grad-weight + grad-input) for stride-2 layers on large maps (fp32, fp16 or bf16 tensors).
//
// Workgroup (channel c, chunk k) walks tiles (image n, band of rows).  Per tile two images are staged
// in LDS: the band of x the grad-weight sums need, and the (four times smaller) band of gy.  A lane
// owns BQ x 2 elements of gy:
//   grad-input : out[2q + r] = sum_a gy[q - m + r + a] * rot'[r + 2a] along each axis (the zero-stuffed
//                gradient never exists); the lane's 2*BQ x 4 block of gx goes straight to memory
//                with 128-bit stores that are contiguous across lanes;
//   grad-weight: its gy elements (the centre of the window it just walked) against the x window
//                they touch, accumulated in K*K registers for the whole chunk, then reduced in a fixed
//                order exactly like the stride-1 kernel (DPP within a wavefront, LDS across
//                wavefronts) into partial[c][k][tap].
// gy is read from HBM once for both gradients; the reference reads it twice
// (torch_dwconv/dwconv.py:56-68) and x K*K times (torch_dwconv/dwconv_kernel.cu:260-306).
#include "dwconv_tile_common.hpp"

#include <type_traits>

namespace dwconv {

namespace {

// Both images of a tile.  At 36 KiB the 5x5 kernels on 75- to 80-wide maps get one band more, which is nearly empty: bf16,
// batch 64, 75x75 C=144 219 us against 162 at 40 KiB, 80x80 106 / 80; fp32 75x75 148 / 138; every other layer of 185- to
// 320-pixel EfficientNets within 2 %.  48 KiB leaves three workgroups per CU: 117x117 C=96 3x3 5 % slower.
constexpr int kFusedLdsBudget = 40 * 1024;

struct BwdS2Plan {
    StageLayout sx;   // x image: row r holds x row 2*q0 - pad + r, column c holds x column c - pad
    StageLayout sg;   // gy image: row r holds gy row q0 - m + r, column c holds gy column c - m
    const void *x;    // element type IO of the kernel template
    const void *gy;
    const void *taps;
    void *gx;
    float *partial;
    int channel;
    int pad;          // forward padding (both axes)
    int m;            // (K - 1 - pad + E) / 2
    int g_base;       // float offset of the gy image in LDS
    int rows_per_tile;  // half-resolution rows per tile
    int row_tiles;
    int tiles_per_group, chunks;
    int ncb;
    unsigned ncb_magic;
    int n_items;
    int bq;
    int vec_gx;
    bool prefetch;    // two-step staging, if the tensors turn out to be reachable through buffer views
    int out_h, out_w; // extent of gy (the epilogue's instances)
    EpilogueBackward epi;
};


// E = parity of the transposed problem's leading pad K - 1 - pad (the same on both axes).
// BQ: half-resolution rows per lane (4; 2 for planes too low to give every lane a block of 4).
// VIEWS: x, gy and gx all go through buffer views (sx.vec_in == sg.vec_in == vec_gx == 2), nothing else compiled in.
// PF: the images travel in two steps (fetch_rows / commit_rows; without VIEWS their forms for 16-bit rows of any width), each
// one's loads in flight during an arithmetic phase.  Order of a tile, two barriers as without PF: [gy of this tile is in registers] commit gy |
// barrier | issue the loads of x | grad-input from the gy windows | commit x | barrier | issue the loads of the next
// tile's gy | grad-weight sums over the x windows.
// EPI (padding K/2): gy is the gradient of act(conv * scale + shift).  The x image covers every gy row that a tile's in_grad
// depends on, K/2 more than its own, so each lane recomputes the convolution of a BQ x 2 block of them and replaces gy in LDS
// by the gradient of the convolution; two more sums are the gradients of scale and shift.  A tile is units * BQ - K/2 rows, and
// the last lanes of a column take the last BQ of them, of which they own those no other lane has.
constexpr int kPrefetchSlots = 8;  // loads per lane and image at most (the planner checks rows_fit)

template <typename IO, int K, int E, int BQ, bool VIEWS, bool PF = false, bool EPI = false>
__global__ __launch_bounds__(kThreads) void bwd_s2_kernel(const BwdS2Plan p)
{
    extern __shared__ float4 lds_raw[];
    float *lds = reinterpret_cast<float *>(lds_raw);
    const IO *const x = static_cast<const IO *>(p.x);
    const IO *const gy = static_cast<const IO *>(p.gy);
    constexpr int KK = K * K;
    constexpr int KA = (K + E + 1) / 2;
    constexpr int GW_ROWS = BQ + KA;                  // gy window rows
    constexpr int NWG = 2 * ((KA + 2 + 1) / 2);       // gy window columns, as float2s
    constexpr int XW_ROWS = (BQ - 1) * 2 + K;         // x window rows
    constexpr int NVX = (K + 2 + 3) / 4;              // x window columns, as float4s

    // every XCD (own L2) gets a contiguous run of workgroups: chunks k and k + 1 of a channel walk neighbouring
    // bands in step and share their halo rows (-2 % on the 112x112 layer)
    const int wg = xcd_contiguous_tile(blockIdx.x, gridDim.x);
    const int c = wg / p.chunks;
    const int chunk = wg - c * p.chunks;

    const bool has_item = static_cast<int>(threadIdx.x) < p.n_items;
    const int item = has_item ? threadIdx.x : 0;
    const int rb = fast_div(item, p.ncb_magic);
    const int cb = item - rb * p.ncb;
    static_assert(!EPI || !PF, "the epilogue's instances stage in one step");
    constexpr int M = (K - 1 - K / 2 + E) / 2;  // p.m of the epilogue's instances
    EpilogueSums sums;
    float e_scale = 1.f, e_shift = 0.f;
    if constexpr (EPI) p.epi.load(c, e_scale, e_shift);

    float rot[KK];
#pragma unroll
    for (int t = 0; t < KK; ++t) rot[t] = Io<IO>::in(static_cast<const IO *>(p.taps)[c * KK + KK - 1 - t]);
    float wacc[KK];
#pragma unroll
    for (int t = 0; t < KK; ++t) wacc[t] = 0.f;

    // (rows of any width: 16-bit elements only, three dwords a slot)
    constexpr bool PF_ANY = PF && !VIEWS;
    RowLane lane_x{}, lane_g{};
    typename std::conditional<PF_ANY, unsigned[3], typename Raw4<IO>::type>::type staged[PF ? kPrefetchSlots : 1];
    auto fetch = [&](const StageLayout &s, const RowLane &l, const IO *plane, int iy0) {
        if constexpr (PF_ANY) fetch_rows_any<IO, kPrefetchSlots>(s, l, plane, iy0, staged);
        else if constexpr (PF) fetch_rows<IO, kPrefetchSlots>(s, l, plane, iy0, staged);
    };
    auto commit = [&](const StageLayout &s, const RowLane &l, const IO *plane, int iy0, float *image) {
        if constexpr (PF_ANY) commit_rows_any<IO, kPrefetchSlots>(s, l, plane, iy0, image, staged);
        else if constexpr (PF) commit_rows<IO, kPrefetchSlots>(s, l, image, staged);
    };
    if constexpr (PF) {
        lane_x = row_lane<IO>(p.sx);
        lane_g = row_lane<IO>(p.sg);
        if (chunk < p.tiles_per_group) {
            const int n = chunk / p.row_tiles, rt = chunk - n * p.row_tiles;
            fetch(p.sg, lane_g, gy + (static_cast<long>(n) * p.channel + c) * p.sg.in_plane, rt * p.rows_per_tile - p.m);
        }
    }

    for (int tile = chunk; tile < p.tiles_per_group; tile += p.chunks) {
        const int n = tile / p.row_tiles, rt = tile - n * p.row_tiles;
        const long plane0 = static_cast<long>(n) * p.channel + c;
        const int q0 = rt * p.rows_per_tile;
        // The first gy row of this lane's block in the tile, and how many of its first rows belong to another lane.  (With the epilogue
        // the last blocks end with the band and the plane, as in wgrad_tile_kernel: no row past the plane meets x.)
        const int qb = EPI ? max(min(rb * BQ, min(p.rows_per_tile, p.out_h - q0) - BQ), 0) : rb * BQ;
        const int skip = EPI ? rb * BQ - qb : 0;
        // (the epilogue's x image starts at the window of gy row q0 - M + E, the first one that in_grad depends on)
        const float *base_x = lds + ((EPI ? qb + M - E : qb) * 2) * p.sx.pitch + kSlack + 4 * cb;
        const float *base_g = lds + p.g_base + qb * p.sg.pitch + kSlack + 2 * cb;

        if constexpr (PF) {
            // (every lane read its gy windows of the previous tile before that tile's second barrier)
            commit(p.sg, lane_g, gy + plane0 * p.sg.in_plane, q0 - p.m, lds + p.g_base);
            __syncthreads();
            fetch(p.sx, lane_x, x + plane0 * p.sx.in_plane, 2 * q0 - p.pad);
        } else {
            if (tile != chunk) __syncthreads();  // the previous tile's window reads are done
            // fp32: two 16-byte loads in flight per lane and image (not four): -3 % on the 112x112 layer, the two
            // images' loads overlap.  16-bit elements: four 8-byte loads, the same bytes in flight (112x112 C=96
            // 176 -> 166 us).
            constexpr int kInFlight = sizeof(IO) == 2 ? 4 : 2;
            stage_tile<IO, VIEWS, kInFlight>(p.sx, x, lds, plane0, 1, 2 * (EPI ? q0 - M + E : q0) - p.pad);
            stage_tile<IO, VIEWS, kInFlight>(p.sg, gy, lds + p.g_base, plane0, 1, q0 - p.m);
            __syncthreads();
        }

        if constexpr (EPI) {
            float z[BQ][2];
#pragma unroll
            for (int b = 0; b < BQ; ++b) z[b][0] = z[b][1] = 0.f;
            const float *xw = lds + (rb * BQ * 2) * p.sx.pitch + kSlack + 4 * cb;
            float nxt[4 * NVX];
            load_window_row<NVX>(xw, nxt);
#pragma unroll
            for (int wr = 0; wr < XW_ROWS; ++wr) {
                float win[4 * NVX];
#pragma unroll
                for (int i = 0; i < 4 * NVX; ++i) win[i] = nxt[i];
                if (wr + 1 < XW_ROWS) load_window_row<NVX>(xw + (wr + 1) * p.sx.pitch, nxt);
#pragma unroll
                for (int b = 0; b < BQ; ++b) {
                    const int ty = wr - 2 * b;
                    if (ty < 0 || ty >= K) continue;
#pragma unroll
                    for (int tx = 0; tx < K; ++tx)
#pragma unroll
                        for (int o = 0; o < 2; ++o) z[b][o] = fmaf(win[2 * o + tx], rot[KK - 1 - (ty * K + tx)], z[b][o]);
                }
                pin_registers(z);
            }
            float *gp = lds + p.g_base + (rb * BQ + E) * p.sg.pitch + kSlack + 2 * cb + M;
            float s_scale = 0.f, s_shift = 0.f;
            p.epi.slopes(z, e_scale, e_shift, [&](auto act) {
#pragma unroll
                for (int b = 0; b < BQ; ++b) {
                    const int r = rb * BQ + b + E - M;  // row of the tile
                    const bool row_ok = has_item && static_cast<unsigned>(q0 + r) < static_cast<unsigned>(p.out_h);
                    const bool own = row_ok && static_cast<unsigned>(r) < static_cast<unsigned>(p.rows_per_tile);
#pragma unroll
                    for (int o = 0; o < 2; ++o) {
                        const bool col_ok = 2 * cb + o < p.out_w;
                        const float ga = EpilogueBackward::slope<decltype(act)::value>(fmaf(z[b][o], e_scale, e_shift), gp[b * p.sg.pitch + o]);
                        s_scale = fmaf(own && col_ok ? ga : 0.f, own && col_ok ? z[b][o] : 0.f, s_scale);
                        s_shift += own && col_ok ? ga : 0.f;
                        if (row_ok && col_ok) gp[b * p.sg.pitch + o] = ga * e_scale;
                    }
                }
            });
            sums.add(s_scale, s_shift);
            __syncthreads();
        }

        // ---- gy window: grad-input block, and this lane's gy elements from the window's centre
        float g[BQ][2];
        float xacc[2 * BQ][4];
#pragma unroll
        for (int b = 0; b < 2 * BQ; ++b)
#pragma unroll
            for (int o = 0; o < 4; ++o) xacc[b][o] = 0.f;
        float nxg[NWG];
        load_window_row2<NWG / 2>(base_g, nxg);
#pragma unroll
        for (int wr = 0; wr < GW_ROWS; ++wr) {
            float win[NWG];
#pragma unroll
            for (int i = 0; i < NWG; ++i) win[i] = nxg[i];
            if (wr + 1 < GW_ROWS) load_window_row2<NWG / 2>(base_g + (wr + 1) * p.sg.pitch, nxg);
            if (wr >= p.m && wr - p.m < BQ) {
                // the centre row index depends on m (1 or 2 for the kernels served here): select at run time
#pragma unroll
                for (int bq = 0; bq < BQ; ++bq)
                    if (wr - p.m == bq) {
                        const bool mine = has_item && (!EPI || bq >= skip);
                        g[bq][0] = mine ? (p.m == 1 ? win[1] : (p.m == 2 ? win[2] : win[0])) : 0.f;
                        g[bq][1] = mine ? (p.m == 1 ? win[2] : (p.m == 2 ? win[3] : win[1])) : 0.f;
                    }
            }
#pragma unroll
            for (int bq = 0; bq < BQ; ++bq)
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    const int a = wr - bq - r;
                    if (a < 0 || a >= KA) continue;
                    const int fy = r + 2 * a - E;
                    if (fy < 0 || fy >= K) continue;
#pragma unroll
                    for (int xq = 0; xq < 2; ++xq)
#pragma unroll
                        for (int rx = 0; rx < 2; ++rx)
#pragma unroll
                            for (int ax = 0; ax < KA; ++ax) {
                                const int fx = rx + 2 * ax - E;
                                if (fx < 0 || fx >= K) continue;
                                xacc[2 * bq + r][2 * xq + rx] =
                                    fmaf(win[xq + rx + ax], rot[fy * K + fx], xacc[2 * bq + r][2 * xq + rx]);
                            }
                }
            pin_registers(xacc);
        }
        if constexpr (PF_ANY) {
            // (rows 2 (q0 + qb) + b: every lane's row b starts on the same side of a 32-bit boundary)
            const int ox = 4 * cb;
            const IO *const to = static_cast<IO *>(p.gx) + plane0 * p.sx.in_plane;
            const AnyWidthView wide = any_width_view(to, static_cast<long>(p.sx.in_plane) * 2);
            const bool col_ok = has_item && ox < p.sx.in_w;
#pragma unroll
            for (int b = 0; b < 2 * BQ; ++b) {
                const int oy = 2 * (q0 + qb) + b;
                const bool ok = col_ok && oy < p.sx.in_h;
                const bool odd = ((static_cast<unsigned>(b) * p.sx.in_w) & 1u) != (wide.bias >> 1);
                view_store_any<IO>(wide.view, ok ? (oy * p.sx.in_w + ox) * 2u + wide.bias : kOob, p.sx.in_w - ox, p.sx.in_w & 3, odd,
                                   xacc[b][0], xacc[b][1], xacc[b][2], xacc[b][3]);
            }
        } else if (VIEWS || p.vec_gx >= 2) {
            // branch-free: rows and column blocks past the end of the plane store out of range
            const int ox = 4 * cb;
            const __amdgpu_buffer_rsrc_t view = buffer_view(static_cast<IO *>(p.gx) + plane0 * p.sx.in_plane, static_cast<long>(p.sx.in_plane) * sizeof(IO));  // this plane only
            const bool col_ok = has_item && ox < p.sx.in_w;
            bool done = false;
            if constexpr (!VIEWS) {
                if (p.vec_gx == 3) {  // rows of any width: the block that ends a row may be short
#pragma unroll
                    for (int b = 0; b < 2 * BQ; ++b) {
                        const int oy = 2 * (q0 + qb) + b;
                        const bool ok = col_ok && oy < p.sx.in_h && (!EPI || b >= 2 * skip);
                        view_store_first<IO>(view, ok ? (oy * p.sx.in_w + ox) * static_cast<unsigned>(sizeof(IO)) : kOob,
                                             p.sx.in_w - ox, p.sx.in_w & 3, xacc[b][0], xacc[b][1], xacc[b][2], xacc[b][3]);
                    }
                    done = true;
                }
            }
            if (!done) {
#pragma unroll
                for (int b = 0; b < 2 * BQ; ++b) {
                    const int oy = 2 * (q0 + qb) + b;
                    const bool ok = col_ok && oy < p.sx.in_h && (!EPI || b >= 2 * skip);
                    view_store4<IO>(view, ok ? (oy * p.sx.in_w + ox) * static_cast<unsigned>(sizeof(IO)) : kOob, xacc[b][0],
                                    xacc[b][1], xacc[b][2], xacc[b][3]);
                }
            }
        } else if (!VIEWS && has_item) {
            const int ox = 4 * cb;
            IO *dst = static_cast<IO *>(p.gx) + plane0 * p.sx.in_plane + ox;
#pragma unroll
            for (int b = 0; b < 2 * BQ; ++b) {
                const int oy = 2 * (q0 + qb) + b;
                if (oy >= p.sx.in_h || (EPI && b < 2 * skip)) continue;
                IO *row = dst + static_cast<long>(oy) * p.sx.in_w;
                if (p.vec_gx) {
                    if (ox < p.sx.in_w) store4<IO>(row, xacc[b][0], xacc[b][1], xacc[b][2], xacc[b][3]);
                } else {
#pragma unroll
                    for (int o = 0; o < 4; ++o)
                        if (ox + o < p.sx.in_w) row[o] = Io<IO>::out(xacc[b][o]);
                }
            }
        }

        if constexpr (PF) {
            // (every lane read its x windows of the previous tile before this tile's first barrier)
            commit(p.sx, lane_x, x + plane0 * p.sx.in_plane, 2 * q0 - p.pad, lds);
            __syncthreads();
            const int next = tile + p.chunks;
            if (next < p.tiles_per_group) {
                const int nn = next / p.row_tiles, nrt = next - nn * p.row_tiles;
                fetch(p.sg, lane_g, gy + (static_cast<long>(nn) * p.channel + c) * p.sg.in_plane, nrt * p.rows_per_tile - p.m);
            }
        }

        // ---- x window: grad-weight sums
        float nxx[4 * NVX];
        load_window_row<NVX>(base_x, nxx);
#pragma unroll
        for (int wr = 0; wr < XW_ROWS; ++wr) {
            float win[4 * NVX];
#pragma unroll
            for (int i = 0; i < 4 * NVX; ++i) win[i] = nxx[i];
            if (wr + 1 < XW_ROWS) load_window_row<NVX>(base_x + (wr + 1) * p.sx.pitch, nxx);
#pragma unroll
            for (int bq = 0; bq < BQ; ++bq) {
                const int ty = wr - 2 * bq;
                if (ty < 0 || ty >= K) continue;
#pragma unroll
                for (int tx = 0; tx < K; ++tx)
#pragma unroll
                    for (int o = 0; o < 2; ++o) wacc[ty * K + tx] = fmaf(g[bq][o], win[2 * o + tx], wacc[ty * K + tx]);
            }
            pin_registers(wacc);
        }
    }

    __syncthreads();  // the images are dead; their LDS is reused for the reduction
    constexpr int SUMS = EPI ? KK + 2 : KK;
#pragma unroll
    for (int t = 0; t < SUMS; ++t) {
        const float s = wave_sum_to_last_lane(t < KK ? wacc[t < KK ? t : 0] : static_cast<float>(t == KK ? sums.scale : sums.shift));
        if ((threadIdx.x & 63) == 63) lds[(threadIdx.x >> 6) * SUMS + t] = s;
    }
    __syncthreads();
    if (threadIdx.x < SUMS) {
        float s = lds[threadIdx.x];
        for (int w = 1; w < static_cast<int>(blockDim.x) / 64; ++w) s += lds[w * SUMS + threadIdx.x];
        p.partial[(static_cast<long>(c) * p.chunks + chunk) * SUMS + threadIdx.x] = s;
    }
}

template <int K, bool EPI = false>
bool plan_bwd_s2(BwdS2Plan &p, const WgradGeometry &g, int kBq, size_t esize)
{
    constexpr int HALO = EPI ? K / 2 : 0;  // gy rows of a tile's image block that belong to its neighbours
    const int pad0 = K - 1 - g.pad_h;  // leading pad of the transposed problem
    const int E = pad0 & 1;
    const int KA = (K + E + 1) / 2;
    const int NWG = 2 * ((KA + 2 + 1) / 2);
    const int NVX = (K + 2 + 3) / 4;
    p.channel = g.channel;
    p.bq = kBq;
    p.pad = g.pad_h;
    p.m = (pad0 + E) / 2;
    if (p.m > 2) return false;
    p.ncb = ceil_div(std::max((g.in_w + 1) / 2, g.out_w), 2);
    if (p.ncb > kThreads) return false;

    p.sx.in_h = g.in_h;
    p.sx.in_w = g.in_w;
    p.sx.in_plane = g.in_h * g.in_w;
    p.sx.col_shift = g.pad_w;
    layout_columns(p.sx, 4 * (p.ncb - 1) + 4 * NVX);
    p.sg.in_h = g.out_h;
    p.sg.in_w = g.out_w;
    p.sg.in_plane = g.out_h * g.out_w;
    p.sg.col_shift = p.m;
    layout_columns(p.sg, 2 * (p.ncb - 1) + NWG);

    const int qrows = std::max((g.in_h + 1) / 2, g.out_h);
    p.out_h = g.out_h;
    p.out_w = g.out_w;
    const int min_units = EPI ? 2 : 1;  // (the epilogue's tiles have BQ rows of their own at least)
    const int row_units = std::max(ceil_div(qrows + HALO, kBq), min_units);
    auto rows_x = [&](int units) { return (units * kBq - 1) * 2 + K; };
    auto rows_g = [&](int units) { return units * kBq - HALO + KA; };
    auto bytes = [&](int units) {
        return (static_cast<long>(rows_x(units)) * p.sx.pitch + static_cast<long>(rows_g(units)) * p.sg.pitch) * 4;
    };
    int units = kThreads / p.ncb;
    if (units < min_units) {
        if (EPI) return false;
        units = 1;
    }
    if (units > row_units) units = row_units;
    const int budget = env_int("DWCONV_FUSED_LDS", kFusedLdsBudget);
    // (with the epilogue a plane that fits 48 KiB stays whole: two bands would each leave half of the lanes idle)
    const bool whole = EPI && units == row_units && bytes(units) <= 48 * 1024;
    while (!whole && units > min_units && bytes(units) > budget) --units;
    if (bytes(units) > 60 * 1024) return false;
    int bands;
    if constexpr (EPI) {
        bands = ceil_div(qrows, units * kBq - HALO);
        units = std::max(ceil_div(ceil_div(qrows, bands) + HALO, kBq), min_units);
        bands = ceil_div(qrows, units * kBq - HALO);
    } else {
        bands = ceil_div(row_units, units);
        units = ceil_div(row_units, bands);
    }
    p.rows_per_tile = units * kBq - HALO;
    p.row_tiles = bands;
    if (!layout_rows(p.sx, rows_x(units), 1) || !layout_rows(p.sg, rows_g(units), 1)) return false;
    p.g_base = p.sx.plane_pitch;
    p.n_items = units * p.ncb;
    p.ncb_magic = magic_u16(p.ncb);
    const long tiles = static_cast<long>(g.batch) * bands;
    if (tiles > 0x7fffffffL) return false;
    p.tiles_per_group = static_cast<int>(tiles);
    // Workgroups in all.  The fp32 5x5 / 7x7 kernels gain from twice as many, shorter chunks; the 3x3 one does not, and with 16-bit elements, where the kernel is bound by
    // instruction issue, the per-workgroup prologue and reduction make more chunks 8-15 % slower.
    // Two-step staging (see the kernel) is for 16-bit elements, where the arithmetic is long against the bytes: 56x56
    // 5x5 bf16 88 -> 81 us, 112x112 3x3 bf16 162 -> 156.  It needs several tiles per workgroup, and its registers
    // leave room for four workgroups per CU (three with 7x7 filters), so the workgroups are counted to fill the chip
    // three times over, rounded down (with one chunk more per channel, a fourth, nearly empty round: +5 %).  With fp32
    // elements it gains on some layers and loses on others inside a training step (48x48 5x5 92 -> 85 us, 56x56 117 ->
    // 124, 64x64 137 -> 142; 3x3 112x112 274 -> 287): those kernels wait for memory with all their loads in flight
    // as they are, and stay as they were.  16-bit rows of any width gain more, since a lane's column, its cut at the row's
    // end and its shift are worked out per lane and row instead of per slot, and half of the in_grad rows leave in 64-bit pieces:
    // bf16, batch 64, 150x150 C=96 3x3 235 -> 165 us, 75x75 C=144 5x5 161 -> 113, 38x38 C=240 3x3 84 -> 57.  The choice is made from the geometry alone, so that the workspace query
    // and the launch agree; tensors that then turn out to be misaligned run the one-step kernel on the same chunks.
    const int pf_mode = env_int("DWCONV_S2_PREFETCH", 1);  // 0: never, 1: 16-bit elements, 2: wherever it fits
    const bool whole_groups = g.in_w % 4 == 0 && g.out_w % 4 == 0;
    p.prefetch = !EPI && (pf_mode == 2 || (pf_mode == 1 && esize == 2)) && rows_fit(p.sx, kPrefetchSlots) &&
                 rows_fit(p.sg, kPrefetchSlots) && (whole_groups || (esize == 2 && env_int("DWCONV_S2_PF_ANY", 1))) &&
                 stage_vector_mode(p.sx, 1, esize) == 2 && stage_vector_mode(p.sg, 1, esize) == 2 &&
                 vector_mode(1, p.sx.in_plane, esize) == 2;
    int chunks;
    if (p.prefetch) {
        chunks = env_int("DWCONV_WGRAD_WGS", kCus * (K == 7 ? 3 : 4) * 3) / g.channel;
    } else {
        // (5x5 fp32: 6144 against 12288 measured 3-8 % faster on 48- to 64-wide maps, the same at 75 and 128 x 96;
        // 3x3 fp32: on maps 96 wide and more three workgroups per CU, all resident from the start, against 3072: 2-7 %
        // faster on 96-, 112- and 120-wide layers; 38 x 38 likes twice as many, 129 -> 121 us)
        // (with the epilogue: 112x112 C=96 fp32 352 us with 768, 302 with 6144)
        const int wgs = (K >= 5 && esize == 4) || (EPI && K == 3) ? 6144 : (K == 3 && esize == 4 ? (g.in_w >= 96 ? 768 : (g.in_w < 48 ? 6144 : 3072)) : 3072);
        chunks = ceil_div(env_int(K == 3 ? "DWCONV_S2_WGS_K3" : "DWCONV_WGRAD_WGS", wgs), g.channel);
    }
    if (chunks > p.tiles_per_group) chunks = p.tiles_per_group;
    if (chunks < 1) chunks = 1;
    p.chunks = chunks;
    if (static_cast<long>(g.channel) * chunks > 0x7fffffffL) return false;
    return true;
}

template <typename IO, int K, bool EPI = false>
long bwd_s2_case(int mode, const IO *x, const IO *gy, const IO *taps, IO *gx, IO *gw, void *ws,
                 size_t ws_bytes, const WgradGeometry &g, hipStream_t stream, const EpilogueBackward &epi = {},
                 float *param_grad = nullptr)
{
    constexpr int SUMS = EPI ? K * K + 2 : K * K;
    // blocks of 4 half-resolution rows, or of 2 when that is what it takes to give most lanes an item
    const int qrows = std::max((g.in_h + 1) / 2, g.out_h), pairs = ceil_div(std::max((g.in_w + 1) / 2, g.out_w), 2);
    // (with the epilogue the K/2 rows that a tile shares with its neighbours count: at 64 columns blocks of two would take two
    // bands of 144 lanes where blocks of four take one)
    const int bq = EPI ? (ceil_div(qrows + K / 2, 2) * pairs <= kThreads ? 2 : 4) : (ceil_div(qrows, 4) * pairs * 2 <= kThreads ? 2 : 4);
    BwdS2Plan p{};
    if (!plan_bwd_s2<K, EPI>(p, g, bq, sizeof(IO))) return -1;
    const size_t need = static_cast<size_t>(g.channel) * p.chunks * SUMS * sizeof(float);
    if (mode == 0) return static_cast<long>(need);
    if (ws == nullptr || ws_bytes < need)
        return fail(DWCONV_ERR_WORKSPACE, "backward needs a workspace of %zu bytes, got %zu", need, ws_bytes);
    p.x = x;
    p.gy = gy;
    p.taps = taps;
    p.gx = gx;
    p.partial = static_cast<float *>(ws);
    p.epi = epi;
    p.sx.vec_in = row_vector_mode(g.in_w, x);
    p.sg.vec_in = row_vector_mode(g.out_w, gy);
    p.vec_gx = row_vector_mode(g.in_w, gx, false);
    // (rows of any width, mode 3, need the view; the aligned modes choose between pointer and view)
    const int x_view = stage_vector_mode(p.sx, 1, sizeof(IO)), g_view = stage_vector_mode(p.sg, 1, sizeof(IO));
    const int gx_view = vector_mode(1, p.sx.in_plane, sizeof(IO));
    p.sx.vec_in = p.sx.vec_in == 1 ? x_view : (p.sx.vec_in == 3 && x_view == 2 ? 3 : 0);
    p.sg.vec_in = p.sg.vec_in == 1 ? g_view : (p.sg.vec_in == 3 && g_view == 2 ? 3 : 0);
    p.vec_gx = p.vec_gx == 1 ? gx_view : (p.vec_gx == 3 && gx_view == 2 ? 3 : 0);
    const size_t images = static_cast<size_t>(p.sx.plane_pitch + p.sg.plane_pitch) * 4;
    const size_t red = static_cast<size_t>(kThreads / 64) * SUMS * 4;
    const size_t shmem = images > red ? images : red;
    const int E = (K - 1 - g.pad_h) & 1;
    const dim3 grid(g.channel * p.chunks), block(kThreads)  /* all 256 lanes stage the images even when the tile has fewer items */;
    const bool views = p.sx.vec_in == 2 && p.sg.vec_in == 2 && p.vec_gx == 2 && !env_int("DWCONV_NO_VIEW_ONLY", 0);
    const bool prefetch = views && p.prefetch;
    const bool prefetch_any = !views && p.prefetch && sizeof(IO) == 2 && !env_int("DWCONV_NO_VIEW_ONLY", 0);
    auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, grid, block, shmem, stream, p); };
    auto pick = [&](auto e, auto b) {
        constexpr int kE = decltype(e)::value, kB = decltype(b)::value;
        if constexpr (EPI) {
            if constexpr (kE == ((K - 1 - K / 2) & 1)) {
                if (views) launch(bwd_s2_kernel<IO, K, kE, kB, true, false, true>);
                else launch(bwd_s2_kernel<IO, K, kE, kB, false, false, true>);
            }
        } else if (prefetch) launch(bwd_s2_kernel<IO, K, kE, kB, true, true>);
        else if (prefetch_any) {
            if constexpr (sizeof(IO) == 2) launch(bwd_s2_kernel<IO, K, kE, kB, false, true>);
        }
        else if (views) launch(bwd_s2_kernel<IO, K, kE, kB, true>);
        else launch(bwd_s2_kernel<IO, K, kE, kB, false>);
    };
    using std::integral_constant;
    if (bq == 2) {
        if (E) pick(integral_constant<int, 1>{}, integral_constant<int, 2>{});
        else pick(integral_constant<int, 0>{}, integral_constant<int, 2>{});
    } else if (E) pick(integral_constant<int, 1>{}, integral_constant<int, 4>{});
    else pick(integral_constant<int, 0>{}, integral_constant<int, 4>{});
    const int rc = check_launch("bwd_s2_kernel");
    if (rc != DWCONV_OK) return rc;
    note_variant("bwd_tile_s2%s<k%d,e%d,bq%d%s> rows%d chunks%d vin%d vgy%d vgx%d%s", sizeof(IO) == 2 ? "16" : "", K, E, bq,
                 EPI ? ",epi" : "", p.rows_per_tile, p.chunks, p.sx.vec_in, p.sg.vec_in, p.vec_gx, prefetch || prefetch_any ? " pf" : "");
    if constexpr (EPI) return launch_fused_final(p.partial, gw, param_grad, g.channel, K * K, p.chunks, stream);
    else return launch_wgrad_final(p.partial, gw, g.channel, K * K, p.chunks, stream);
}

// Whether one sweep beats the three calls.  It does with fp32 tensors (0.6 to 0.9 of their time) and with 16-bit ones of few
// elements, where launches count (batch 4, C=144: 0.5 to 0.9).  Else their two-step staging makes up for the extra passes in
// part: time of one sweep to three calls at C = 144, batch 96, bf16, by columns: 3x3 34 1.08, 38 1.08, 40 0.87, 56 0.72, 80 0.90,
// 112 0.91, 150 0.78 (rows of any width, 41 to 106, 0.67 to 0.99, 117 1.09); 5x5 34 1.11, 40 0.97, 48 0.92, 56 0.85, 60 0.90,
// 64 1.10, 75 1.01, 90 1.13, 112 1.20, 150 1.12 (rows of any width, 41 to 59, 0.84 to 1.04, 61 1.29).
bool fused_s2_pays(const WgradGeometry &g, size_t esize)
{
    const long elements = static_cast<long>(g.batch) * g.channel * g.in_h * g.in_w;
    if (esize == 4 || elements < kFusedFewElements || env_int("DWCONV_EPI_ALWAYS", 0)) return true;
    return g.kernel_h == 3 ? g.in_w >= 40 : g.in_w >= 40 && g.in_w < 64;
}

// With the epilogue's backward: padding K/2, filters up to 5x5.
template <typename IO>
long fused_s2_any(int mode, const IO *x, const IO *gy, const IO *taps, IO *gx, IO *gw, float *param_grad, const EpilogueBackward &epi,
                  void *ws, size_t ws_bytes, const WgradGeometry &g, hipStream_t stream)
{
    if (env_int("DWCONV_NO_FUSED_TILE", 0)) return -1;
    const int K = g.kernel_h;
    if (g.kernel_w != K || g.down_h != 2 || g.down_w != 2 || g.dil != 1 || g.mult > 1) return -1;
    if (g.pad_h != K / 2 || g.pad_w != K / 2) return -1;
    if (g.in_h < 1 || g.in_w < 1 || g.out_h != (g.in_h - 1) / 2 + 1 || g.out_w != (g.in_w - 1) / 2 + 1) return -1;
    if (static_cast<long>(g.in_h) * g.in_w >= (1l << 30) || !fused_s2_pays(g, sizeof(IO))) return -1;
    if (K == 3) return bwd_s2_case<IO, 3, true>(mode, x, gy, taps, gx, gw, ws, ws_bytes, g, stream, epi, param_grad);
    if (K == 5) return bwd_s2_case<IO, 5, true>(mode, x, gy, taps, gx, gw, ws, ws_bytes, g, stream, epi, param_grad);
    return -1;
}

template <typename IO>
long bwd_s2_any(int mode, const IO *x, const IO *gy, const IO *taps, IO *gx, IO *gw, void *ws,
                size_t ws_bytes, const WgradGeometry &g, hipStream_t stream)
{
    if (env_int("DWCONV_NO_FUSED_TILE", 0)) return -1;
    const int K = g.kernel_h;
    if (g.kernel_w != K || g.down_h != 2 || g.down_w != 2) return -1;
    if (g.pad_h != g.pad_w || g.pad_h < 0 || g.pad_h > K - 1) return -1;
    if (g.in_h < 1 || g.in_w < 1 || g.out_h < 1 || g.out_w < 1) return -1;
    if (static_cast<long>(g.in_h) * g.in_w >= (1l << 30)) return -1;
    if (K == 3) return bwd_s2_case<IO, 3>(mode, x, gy, taps, gx, gw, ws, ws_bytes, g, stream);
    if (K == 5) return bwd_s2_case<IO, 5>(mode, x, gy, taps, gx, gw, ws, ws_bytes, g, stream);
    if (K == 7) return bwd_s2_case<IO, 7>(mode, x, gy, taps, gx, gw, ws, ws_bytes, g, stream);
    return -1;
}

}  // namespace

size_t bwd_s2_workspace(const WgradGeometry &g)
{
    // partial sums are fp32 whatever the element type, but the number of chunks follows it: the larger of the two plans
    const long n4 = bwd_s2_any<float>(0, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, g, nullptr);
    const long n2 = bwd_s2_any<half_t>(0, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, 0, g, nullptr);
    const long n = std::max(n4, n2);
    return n > 0 ? static_cast<size_t>(n) : 0;
}

template <typename IO>
int try_launch_bwd_s2(const IO *in, const IO *gy, const IO *taps, IO *gx, IO *gw, void *ws, size_t ws_bytes,
                      const WgradGeometry &g, hipStream_t stream)
{
    return static_cast<int>(bwd_s2_any<IO>(1, in, gy, taps, gx, gw, ws, ws_bytes, g, stream));
}

size_t fused_s2_workspace(const WgradGeometry &g, size_t esize)
{
    const EpilogueBackward epi{};
    const long n = esize == 4 ? fused_s2_any<float>(0, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, epi, nullptr, 0, g, nullptr)
                              : fused_s2_any<half_t>(0, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, epi, nullptr, 0, g, nullptr);
    return n > 0 ? static_cast<size_t>(n) : 0;
}

template <typename IO>
int try_launch_fused_s2(const IO *in, const IO *gy, const IO *taps, IO *gx, IO *gw, float *param_grad, const EpilogueBackward &epi,
                        void *ws, size_t ws_bytes, const WgradGeometry &g, hipStream_t stream)
{
    return static_cast<int>(fused_s2_any<IO>(1, in, gy, taps, gx, gw, param_grad, epi, ws, ws_bytes, g, stream));
}

#define DWCONV_INSTANTIATE(IO)                                                                                                 \
    template int try_launch_fused_s2<IO>(const IO *, const IO *, const IO *, IO *, IO *, float *, const EpilogueBackward &,    \
                                         void *, size_t, const WgradGeometry &, hipStream_t);
DWCONV_INSTANTIATE(float)
DWCONV_INSTANTIATE(half_t)
DWCONV_INSTANTIATE(bf16_t)
#undef DWCONV_INSTANTIATE

template int try_launch_bwd_s2<float>(const float *, const float *, const float *, float *, float *, void *, size_t,
                                      const WgradGeometry &, hipStream_t);
template int try_launch_bwd_s2<half_t>(const half_t *, const half_t *, const half_t *, half_t *, half_t *, void *, size_t,
                                       const WgradGeometry &, hipStream_t);
template int try_launch_bwd_s2<bf16_t>(const bf16_t *, const bf16_t *, const bf16_t *, bf16_t *, bf16_t *, void *, size_t,
                                       const WgradGeometry &, hipStream_t);

}  // namespace dwconv
