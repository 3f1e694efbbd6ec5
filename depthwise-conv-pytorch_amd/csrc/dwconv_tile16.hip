// LDS-tiled forward / stride-1 grad-input kernel for 16-bit tensors (fp16, bf16): rows that are whole groups of eight
// elements, and an instance (ANY) for rows of any other width that start on any element.
//
// The tiled kernels of dwconv_tile.hip widen every element to fp32 on its way into LDS.  With 16-bit tensors they
// are bound by the vector unit, not by memory: the same instructions move half the bytes.  This kernel keeps the
// elements as loaded, two per dword:
//   load  = eight elements (16 bytes) per lane and load, written to LDS as they are; a lane keeps its column and
//           walks down the rows, so a slot costs a handful of integer instructions.
//   taps  = packed in pairs (t[2j], t[2j+1]) as the tensor's own 16-bit values.
//   item  = BH x 8 outputs (stride 1) or BH x 4 outputs (stride 2) per lane.  A window row is read as dwords; the
//           pairs that start at an odd element are formed with one v_alignbit each, and every output takes
//           ceil(K/2) two-element dot products (v_dot2c_f32_f16 / v_dot2c_f32_bf16, each as exact as two multiply-adds in fp32) per
//           filter row instead of K multiply-adds.  The last tap of a row has no partner: its element is isolated
//           with a mask (a garbage partner times a zero tap would turn an Inf next to the window into a NaN).
// Same results as the fp32-image kernel up to the order of the fp32 additions.
// Replaces, for these tensors, what torch_dwconv/dwconv_kernel.cu:69-181 computes with `scalar_t` = half.
#include "dwconv_tile16_common.hpp"

namespace dwconv {

namespace {

struct Tile16Plan {
    const void *in;
    const void *taps;
    void *out;
    long planes;
    int channel;
    Image16 im;
    int out_h, out_w, out_plane;
    int pad_h, pad_w;
    int rows_per_tile;     // output rows per tile, a multiple of BH
    int row_tiles;         // tiles per plane
    int planes_per_tile;
    int n_tiles;
    int ncb;               // column blocks per row
    unsigned ncb_magic;
    int items_per_plane;
    unsigned ipp_magic;
    int tap_base;          // dword offset of the tap tables in LDS
    int dump;              // slot index of a spare slot
    int lout;              // results leave through LDS as one linear stream per plane (one item per lane)
    Epilogue epi;
};

// PW1: parity of the left padding (the first element of a lane's window is the high half of a dword when odd).
// EPI: the epilogue of the fused forward entry points is compiled in (its temporaries cost 12 registers, a wavefront
// of occupancy, also when it is switched off at run time).
// ANY: rows of any width at any element alignment, on either side.  The fp32-image kernel, which such rows took before, loads
// four elements at a time (three dwords each where rows start on odd elements), widens them on their way into LDS and takes a
// multiply-add per tap: at 150x150 C=96 3x3 stride 2 the bytes take 56 us and it took 119.  Here a load brings eight elements
// (four dwords, or five), nothing is widened, and the results, whose rows start anywhere too, leave through LDS as one run of
// 16-byte pieces (lds_put_run16, store_run16).  bf16, batch 64, us before / now: 150x150 3x3 C=32 53.4 / 45.8, stride 2 C=96
// 119 / 90; 75x75 C=144 3x3 71.6 / 51.3, 5x5 stride 2 58.8 / 44.3; 38x38 C=240 3x3 stride 2 26.5 / 20.9; 107x107 C=32 3x3
// 33.9 / 27.7, stride 2 C=96 77.9 / 55.6.  What is left is the LDS traffic of the results (five writes a row where an aligned
// one is a single write) and the lines at the ends of a band that two workgroups fetch.
template <typename IO, int K, int S, int PW1, bool FLIP, int BH, bool EPI, bool ANY>
__global__ __launch_bounds__(kThreads) void fir_down16_kernel(const Tile16Plan p)
{
    extern __shared__ float4 lds_raw[];
    uint32_t *lds32 = reinterpret_cast<uint32_t *>(lds_raw);
    constexpr int OWI = S == 1 ? 8 : 4;      // outputs per item and row
    constexpr int KP = (K + 1) / 2;          // tap pairs per filter row
    constexpr int TPP = K * (KP + 1);        // dwords of a plane's tap table: KP pairs and the last tap as (0, t)
    constexpr int WIN_ROWS = (BH - 1) * S + K;
    constexpr int NDW = (PW1 + (OWI - 1) * S + K - 1) / 2 + 1;  // dwords of a window row

    const int tile = xcd_contiguous_tile(blockIdx.x, p.n_tiles);
    const int pg = tile / p.row_tiles, rt = tile - pg * p.row_tiles;
    const long plane0 = static_cast<long>(pg) * p.planes_per_tile;
    const int nplanes = static_cast<int>(min(static_cast<long>(p.planes_per_tile), p.planes - plane0));
    const int oy0 = rt * p.rows_per_tile;
    const int iy0 = oy0 * S - p.pad_h;
    const int c0 = static_cast<int>(plane0 % p.channel);

    // tap tables
    for (int i = threadIdx.x; i < nplanes * TPP; i += blockDim.x) {
        const int pl = i / TPP, t = i - pl * TPP;
        const int ty = t / (KP + 1), j = t - ty * (KP + 1);
        const uint16_t *f = static_cast<const uint16_t *>(p.taps) + ((c0 + pl) % p.channel) * (K * K);
        auto tap = [&](int x) -> uint32_t {
            if (x >= K) return 0u;
            return FLIP ? f[(K - 1 - ty) * K + (K - 1 - x)] : f[ty * K + x];
        };
        lds32[p.tap_base + i] = j < KP ? (tap(2 * j) | (tap(2 * j + 1) << 16)) : (tap(K - 1) << 16);
    }

    stage_image16<IO, 4, ANY>(p.im, static_cast<const IO *>(p.in) + plane0 * p.im.in_plane, lds32, p.dump, nplanes, iy0);
    __syncthreads();

    const int n_items = nplanes * p.items_per_plane;
    const __amdgpu_buffer_rsrc_t oview =
        buffer_view(static_cast<IO *>(p.out) + plane0 * p.out_plane, static_cast<long>(nplanes) * p.out_plane * sizeof(IO));
    // the BH x OWI sums of one item, after the epilogue
    auto convolve = [&](int pl, int rb, int cb, float(&acc)[BH][OWI]) {
        uint32_t tp[K][KP + 1];
#pragma unroll
        for (int ty = 0; ty < K; ++ty)
#pragma unroll
            for (int j = 0; j <= KP; ++j) tp[ty][j] = lds32[p.tap_base + pl * TPP + ty * (KP + 1) + j];

        // the first filter row's last tap as fp32: its product starts every sum (a plain multiply needs no zeroed
        // accumulator, which the accumulating dot product would)
        const float t0_last = Io<IO>::in(__builtin_bit_cast(IO, static_cast<uint16_t>(tp[0][KP] >> 16)));
        // The lane's window starts at logical dword 4 * cb + PH of image row rb * BH * S (pad_w = K / 2 puts its first
        // element (K/2 + PW1) / 2 dwords left of the lane's block, which starts at dword 4 + 4 * cb); window dword i is
        // LDS dword base[swz(PH + i)].
        constexpr int PH = 4 - (K / 2 + PW1) / 2;
        const uint32_t *base = lds32 + __mul24(pl, p.im.pp) + __mul24(rb * BH * S, p.im.rp) + 5 * cb;
        const int rpitch = p.im.rp;  // dwords per image row
        // (no zero fill: the first product of every sum starts from the constant, see below)
        // window rows are read one ahead of their use, into alternating registers, and the sums pinned after every
        // row (see pin_registers)
        uint32_t win[2][NDW];
#pragma unroll
        for (int i = 0; i < NDW; ++i) win[0][i] = base[swz(PH + i)];
#pragma unroll
        for (int wr = 0; wr < WIN_ROWS; ++wr) {
            const uint32_t(&d)[NDW] = win[wr & 1];
            if (wr + 1 < WIN_ROWS) {
#pragma unroll
                for (int i = 0; i < NDW; ++i) win[(wr + 1) & 1][i] = base[(wr + 1) * rpitch + swz(PH + i)];
            }
            // pairs that start at an odd element
            uint32_t q[NDW];
#pragma unroll
            for (int i = 0; i + 1 < NDW; ++i) q[i] = __builtin_amdgcn_alignbit(d[i + 1], d[i], 16);
            // the element under the last tap of each output: alone in its half for the dot product, and as fp32 for
            // the output row this window row starts
            uint32_t last[OWI];
            float lastf[OWI];
#pragma unroll
            for (int o = 0; o < OWI; ++o) {
                const int e = PW1 + o * S + K - 1;
                last[o] = (e & 1) ? (d[e >> 1] & 0xffff0000u) : (d[e >> 1] & 0x0000ffffu);
                const uint16_t h = static_cast<uint16_t>((e & 1) ? d[e >> 1] >> 16 : d[e >> 1] & 0xffffu);
                lastf[o] = Io<IO>::in(__builtin_bit_cast(IO, h));
            }
#pragma unroll
            for (int b = 0; b < BH; ++b) {
                const int ty = wr - b * S;
                if (ty < 0 || ty >= K) continue;
#pragma unroll
                for (int o = 0; o < OWI; ++o) {
                    const int el = PW1 + o * S + K - 1;
                    if (ty == 0) acc[b][o] = lastf[o] * t0_last;
                    else acc[b][o] = dot2<IO>(last[o], (el & 1) ? tp[ty][KP] : tp[ty][KP - 1], acc[b][o]);
#pragma unroll
                    for (int j = 0; j < K / 2; ++j) {
                        const int e = PW1 + o * S + 2 * j;
                        acc[b][o] = dot2<IO>((e & 1) ? q[e >> 1] : d[e >> 1], tp[ty][j], acc[b][o]);
                    }
                }
            }
#pragma unroll
            for (int b = 0; b < BH; ++b)
                if (b * S <= wr) pin_registers(acc[b]);  // the rows that have been started
        }

        if constexpr (EPI) epilogue_apply_block<1>(acc, p.epi, (c0 + pl) % p.channel);
    };
    // a row of sums as packed 16-bit elements
    auto pack_row = [](const float(&a)[OWI], uint32_t(&t)[OWI / 2]) {
#pragma unroll
        for (int i = 0; i < OWI / 2; ++i) {
            if constexpr (std::is_same<IO, bf16_t>::value) t[i] = bf16_pack2(a[2 * i], a[2 * i + 1]);
            else t[i] = f16_pack2(a[2 * i], a[2 * i + 1]);
        }
    };

    if (ANY || p.lout) {
        // One item per lane (the planner guarantees it).  The packed sums go back into LDS in the layout the band has
        // in memory, over the image, and leave as one linear stream per plane: 16 bytes per lane, 1 KiB of
        // consecutive bytes per wavefront and store.  Lane-owned blocks write a row segment at a time; where a row is
        // not a whole number of 128-byte lines (56 elements: 112 bytes) their streaming stores leave partial lines.
        const bool has_item = static_cast<int>(threadIdx.x) < n_items;
        const int item = has_item ? threadIdx.x : 0;
        const int pl = fast_div(item, p.ipp_magic);
        const int rem = item - __mul24(pl, p.items_per_plane);
        const int rb = fast_div(rem, p.ncb_magic);
        const int cb = rem - __mul24(rb, p.ncb);
        const int rows_here = min(p.rows_per_tile, p.out_h - oy0);
        const int run = rows_here * p.out_w;  // elements per plane (a multiple of eight unless ANY)
        // Wavefronts with no item at all skip the arithmetic; lanes without one in the others compute item 0 again.
        // The sums never leave the arm that makes them (merged with the arm that has none, every sum would be zeroed
        // first); what leaves it are the packed rows, and every wavefront meets the one barrier after the branch.
        uint32_t packed[BH][OWI / 2];
#pragma unroll
        for (int b = 0; b < BH; ++b)
#pragma unroll
            for (int i = 0; i < OWI / 2; ++i) packed[b][i] = 0u;
        if (__builtin_amdgcn_readfirstlane(threadIdx.x) < n_items) {
            float acc[BH][OWI];
            convolve(pl, rb, cb, acc);
#pragma unroll
            for (int b = 0; b < BH; ++b) pack_row(acc[b], packed[b]);
        }
        __syncthreads();  // every window has been read: the image can be overwritten
        if constexpr (ANY) {
            // (a tile of several planes holds whole ones: its results are one run too)
            IO *to = static_cast<IO *>(p.out) + plane0 * p.out_plane + static_cast<long>(oy0) * p.out_w;
            const int head = run_head(to);
            uint16_t *image = reinterpret_cast<uint16_t *>(lds_raw);
            if (has_item) {
#pragma unroll
                for (int b = 0; b < BH; ++b)
                    if (rb * BH + b < rows_here)
                        lds_put_run16(image, head + __mul24(pl, p.out_plane) + __mul24(rb * BH + b, p.out_w) + cb * OWI, p.out_w - cb * OWI, packed[b]);
            }
            __syncthreads();
            store_run16(to, image, head, (nplanes - 1) * p.out_plane + run);
            return;
        }
        if (has_item) {
#pragma unroll
            for (int b = 0; b < BH; ++b) {
                if (rb * BH + b < rows_here) {
                    // (one 128- or 64-bit write per lane at a multiple of its size: conflict-free)
                    uint32_t *d = lds32 + ((__mul24(pl, run) + __mul24(rb * BH + b, p.out_w) + cb * OWI) >> 1);
                    if constexpr (OWI == 8) {
                        u32x4 v;
                        v.x = packed[b][0]; v.y = packed[b][1]; v.z = packed[b][2]; v.w = packed[b][3];
                        *reinterpret_cast<u32x4 *>(d) = v;
                    } else {
                        u32x2 v;
                        v.x = packed[b][0]; v.y = packed[b][1];
                        *reinterpret_cast<u32x2 *>(d) = v;
                    }
                }
            }
        }
        __syncthreads();
        const u32x4 *image = reinterpret_cast<const u32x4 *>(lds_raw);
        const int run8 = run >> 3;
        for (int q = 0; q < nplanes; ++q) {
            const unsigned o0 = (__mul24(q, p.out_plane) + __mul24(oy0, p.out_w)) * 2u;
            for (int i = threadIdx.x; i < run8; i += blockDim.x)
                __builtin_amdgcn_raw_buffer_store_b128(image[q * run8 + i], oview, o0 + i * 16u, 0, kStoreStreaming);
        }
        return;
    }

    if constexpr (!ANY) for (int item = threadIdx.x; item < n_items; item += blockDim.x) {
        const int pl = fast_div(item, p.ipp_magic);
        const int rem = item - __mul24(pl, p.items_per_plane);
        const int rb = fast_div(rem, p.ncb_magic);
        const int cb = rem - __mul24(rb, p.ncb);
        float acc[BH][OWI];
        convolve(pl, rb, cb, acc);
        // branch-free: rows past the end of the plane store out of range
        const unsigned o0 = (__mul24(pl, p.out_plane) + cb * OWI) * 2u;
#pragma unroll
        for (int b = 0; b < BH; ++b) {
            const int oy = oy0 + rb * BH + b;
            const unsigned off = oy < p.out_h ? o0 + __mul24(oy, p.out_w) * 2u : kOob;
            uint32_t t[OWI / 2];
            pack_row(acc[b], t);
            if constexpr (OWI == 8) {
                u32x4 v;
                v.x = t[0]; v.y = t[1]; v.z = t[2]; v.w = t[3];
                __builtin_amdgcn_raw_buffer_store_b128(v, oview, off, 0, kStoreStreaming);
            } else {
                u32x2 v;
                v.x = t[0]; v.y = t[1];
                __builtin_amdgcn_raw_buffer_store_b64(v, oview, off, 0, kStoreStreaming);
            }
        }
    }
}

template <typename IO, int K, int S, int PW1, bool FLIP, int BH, bool ANY>
int launch_down16(Tile16Plan &p, hipStream_t stream)
{
    constexpr int OWI = S == 1 ? 8 : 4;
    constexpr int KP = (K + 1) / 2;
    constexpr int TPP = K * (KP + 1);
    const int threads = kThreads;
    const int target_items = env_int("DWCONV_TILE16_ITEMS", threads);
    // (ANY, stride 2: 150x150 C=96 3x3 98 us with 32 KiB, 91 with 40, 88 with 48, but 75x75 C=144 5x5 46, 46 and 54)
    const int budget = env_int("DWCONV_TILE16_LDS", S == 2 ? (ANY ? 40 : 32) * 1024 : 24 * 1024);

    p.ncb = ceil_div(p.out_w, OWI);
    // elements of a row the windows touch: up to input column (ncb * OWI - 1) * S - pad_w + K - 1, and its pair partner
    const int last_col = (p.ncb * OWI - 1) * S - p.pad_w + K;
    layout_image16(p.im, last_col);
    auto rows_for = [](int units) { return (units * BH - 1) * S + K; };
    auto bytes = [&](int units, int planes) {
        return static_cast<long>(planes) * (static_cast<long>(rows_for(units)) * p.im.rp * 4 + TPP * 4) + 20;
    };

    const int row_units = ceil_div(p.out_h, BH);
    const int ipp_full = row_units * p.ncb;
    int units_per_tile = 0, planes_per_tile = 0;
    if (2 * ipp_full <= target_items) {
        units_per_tile = row_units;
        planes_per_tile = target_items / ipp_full;
        while (planes_per_tile > 1 && bytes(units_per_tile, planes_per_tile) > budget) --planes_per_tile;
        if (static_cast<long>(planes_per_tile) > p.planes) planes_per_tile = static_cast<int>(p.planes);
        if (bytes(units_per_tile, planes_per_tile) > budget) planes_per_tile = 0;
    }
    if (planes_per_tile == 0) {
        planes_per_tile = 1;
        units_per_tile = std::max(1, std::min(row_units, target_items / p.ncb));
        while (units_per_tile > 1 && bytes(units_per_tile, 1) > budget) --units_per_tile;
        if (bytes(units_per_tile, 1) > budget) return -1;
        units_per_tile = ceil_div(row_units, ceil_div(row_units, units_per_tile));  // even out the bands
    }
    p.planes_per_tile = planes_per_tile;
    p.rows_per_tile = units_per_tile * BH;
    p.row_tiles = ceil_div(row_units, units_per_tile);
    if (!finish_image16(p.im, rows_for(units_per_tile), planes_per_tile)) return -1;
    p.items_per_plane = units_per_tile * p.ncb;
    if (planes_per_tile * p.items_per_plane >= 65536) return -1;  // 16-bit reciprocals
    if (static_cast<long>(planes_per_tile) * p.out_plane * 2 >= static_cast<long>(kOob)) return -1;
    p.ncb_magic = magic_u16(p.ncb);
    p.ipp_magic = magic_u16(p.items_per_plane);
    p.dump = planes_per_tile * p.im.lds_rows * (p.im.pitch / 8);
    p.tap_base = 5 * (p.dump + 1);
    const long tiles = ceil_div(p.planes, static_cast<long>(planes_per_tile)) * p.row_tiles;
    if (tiles > 0x7fffffffL) return -1;
    p.n_tiles = static_cast<int>(tiles);
    p.lout = env_int("DWCONV_T16_LOUT", 1) && planes_per_tile * p.items_per_plane <= threads &&
             (p.rows_per_tile * p.out_w) % 8 == 0 && p.out_plane % 8 == 0;
    size_t lds = static_cast<size_t>(p.tap_base) * 4 + static_cast<size_t>(planes_per_tile) * TPP * 4;
    if (ANY) {
        if (planes_per_tile * p.items_per_plane > threads) return -1;
        // the run of results takes the place of the image (and of the taps): seven elements in front, whole 16-byte pieces
        const size_t run = (static_cast<size_t>(planes_per_tile - 1) * p.out_plane + static_cast<size_t>(p.rows_per_tile) * p.out_w + 7 + 8) * 2;
        lds = std::max(lds, run);
        if (planes_per_tile > 1 && p.row_tiles != 1) return -1;
    }

    if (!FLIP && p.epi.enabled())
        hipLaunchKernelGGL((fir_down16_kernel<IO, K, S, PW1, FLIP, BH, !FLIP, ANY>), dim3(p.n_tiles), dim3(threads), lds, stream, p);
    else
        hipLaunchKernelGGL((fir_down16_kernel<IO, K, S, PW1, FLIP, BH, false, ANY>), dim3(p.n_tiles), dim3(threads), lds, stream, p);
    note_variant("tile_down16_dot2<k%d,s%d,%s,bh%d> P%d rows%d%s", K, S, FLIP ? "rot" : "fwd", BH, p.planes_per_tile, p.rows_per_tile,
                 ANY ? " runout anywidth" : p.lout ? " ldsout" : "");
    return check_launch("fir_down16_kernel");
}

template <typename IO, int K, int S, bool FLIP>
int launch_down16_parity(Tile16Plan &p, bool any, hipStream_t stream)
{
    const int forced = env_int("DWCONV_TILE_BH", 0);
    const bool seven = forced ? forced == 7 : (p.out_h % 7 == 0 || p.out_h > 64) && p.out_h % 4 != 0;
    constexpr int PW1 = (K / 2) & 1;  // the left padding is K / 2
    if (any) return launch_down16<IO, K, S, PW1, FLIP, 4, true>(p, stream);
    return seven ? launch_down16<IO, K, S, PW1, FLIP, 7, false>(p, stream) : launch_down16<IO, K, S, PW1, FLIP, 4, false>(p, stream);
}

// From how many elements of input on calls on rows of any width come here.  A call of a few workgroups a compute unit lasts about as
// long as one of them, and one lasts longer here: more planes, loads to shift, the results through LDS.  Time here over that of the
// kernels before (fp32 images; stacked for 5x5 and 7x7 on even rows), geometric means over 1659 layers of 33 to 257 columns, by millions
// of elements (single layers lie up to 0.15 to either side):
//                                          -0.6  -0.85   -1.2   -1.7   -2.4   -3.3   -4.7   -6.5   more
//   stride 1, 3x3, odd rows                  1.08   1.05   1.01   1.00   0.98   1.00   0.94   0.89   0.78
//             3x3, even                      1.32   1.28   1.19   1.24   1.23   1.15   1.19   1.04   0.90
//             5x5, odd                       1.06   1.06   0.98   1.03   0.99   1.02   0.97   0.92   0.86
//             5x5, even                      1.37   1.32   1.23   1.20   1.24   1.12   1.14   0.99   0.88
//             7x7, odd                       1.05   1.03   0.96   1.00   1.00   0.92   0.86   0.82   0.77
//             7x7, even                      1.20   1.18   1.07   1.00   1.03   1.02   0.92   0.89   0.85
//   stride 2, 3x3, odd, and even below 128   1.11   1.10   1.07   1.01   1.02   1.01   0.98   0.92   0.85
//             3x3, even from 128 on          1.02   1.03   1.01   0.97   0.93   0.96   0.97   0.94   0.78
//             5x5, below 128                 1.06   1.06   1.02   0.97   1.00   0.98   0.94   0.90   0.83
//             5x5, from 128 on               0.92   0.93   0.90   0.89   0.86   0.94   0.91   0.82   0.68
//             7x7, even below 128            1.05   1.03   0.99   0.95   0.98   0.95   0.85   0.80   0.74
//             7x7, the others                0.92   0.91   0.90   0.90   0.92   0.88   0.82   0.72   0.63
int any_width_least_elements(int K, int S, int w)
{
    const bool even = w % 2 == 0, wide = w >= 128;
    if (S == 1) return even ? (K == 7 ? 1 << 21 : 5 << 20) : (K == 7 ? 1 << 20 : 3 << 19);
    if (K == 3) return even && wide ? 0 : 3 << 19;
    return wide || (K == 7 && !even) ? 0 : 1 << 20;
}

}  // namespace

// -1 when the kernel does not cover g (the caller goes on to the fp32-image kernel).
template <typename IO>
int try_launch_fir_tiled16(const IO *in, const IO *taps, IO *out, const Geometry &g, hipStream_t stream)
{
    static_assert(sizeof(IO) == 2, "16-bit element types");
    if (!env_int("DWCONV_TILE16", 1)) return -1;
    const int K = g.kernel_h, S = g.down_h;
    if (g.kernel_w != K || (K != 3 && K != 5 && K != 7)) return -1;
    if (g.up_h != 1 || g.up_w != 1 || g.down_w != S || (S != 1 && S != 2)) return -1;
    if (S == 2 && !g.forward) return -1;
    // (the window's place within its LDS slots is a compile-time constant: left padding K/2 only)
    if (g.pad_h0 < 0 || g.pad_h0 > 7 || g.pad_w0 != K / 2) return -1;
    if (g.in_h < 1 || g.out_w < 1) return -1;
    // whole groups of eight that start on 16-byte boundaries, or rows of any width at any element alignment
    const bool any = g.in_w % 8 != 0 || g.out_w % (S == 1 ? 8 : 4) != 0 || reinterpret_cast<uintptr_t>(in) % 16 != 0 ||
                     reinterpret_cast<uintptr_t>(out) % 16 != 0;
    // Input rows of at least 48 elements at stride 2 and 72 at stride 1: measured against the fp32-image and stacked
    // kernels on 48 ... 88 wide maps (batch 64, C = 144, bf16 and fp16), stride 2 is 3-29 % faster here at every
    // width, stride 1 6-19 % from 72 on (88 x 88 5x5: equal) and mixed below (56 x 56 3x3 and 7x7: 8-12 % slower;
    // narrower planes have too few 8-wide blocks to occupy the lanes).
    // Rows of any width, measured against the fp32-image kernel on 26 widths from 33 to 257 (batch 16, bf16 and fp16): stride 2
    // is 2-38 % faster here at every width.  At stride 1 rows of an odd width are 2-25 % faster with 3x3 and 5x5 filters from 65
    // columns on (below, 33 to 57: between 20 % faster and 8 % slower), even ones that are no multiple of four 5-13 % from 128 on
    // (below: 7 % faster to 16 % slower, as the lanes fill), and multiples of four, which that kernel loads aligned, are up to
    // 25 % slower (92: 14.2 us there, 18.0 here).  With 7x7 filters every width from 56 on that is no multiple of four is 6-37 %
    // faster.  Small calls stay with the kernels of before: any_width_least_elements.
    if (any) {
        const bool odd = (g.in_w & 1) != 0, four = g.in_w % 4 == 0;
        const int least = S == 2 ? 33 : four ? 1 << 30 : K == 7 ? 56 : odd ? 65 : 128;
        if (g.in_w < env_int("DWCONV_T16_ANY_MIN_W", least)) return -1;
        const long elements = static_cast<long>(g.planes()) * g.in_h * g.in_w;
        if (elements < env_int("DWCONV_T16_ANY_MIN", any_width_least_elements(K, S, g.in_w))) return -1;
    } else if (g.in_w < env_int("DWCONV_T16_MIN_W", S == 2 ? 48 : 72)) {
        return -1;
    }
    if (static_cast<long>(g.in_h) * g.in_w >= (1l << 30) || static_cast<long>(g.out_h) * g.out_w >= (1l << 30)) return -1;

    Tile16Plan p{};
    p.in = in;
    p.taps = taps;
    p.out = out;
    p.planes = g.planes();
    p.channel = g.channel;
    p.epi = g.epi;
    p.im.in_h = g.in_h;
    p.im.in_w = g.in_w;
    p.im.in_plane = g.in_h * g.in_w;
    p.out_h = g.out_h;
    p.out_w = g.out_w;
    p.out_plane = g.out_h * g.out_w;
    p.pad_h = g.pad_h0;
    p.pad_w = g.pad_w0;
    const bool rot = !g.forward;
    if (S == 1) {
        if (K == 3) return rot ? launch_down16_parity<IO, 3, 1, true>(p, any, stream) : launch_down16_parity<IO, 3, 1, false>(p, any, stream);
        if (K == 5) return rot ? launch_down16_parity<IO, 5, 1, true>(p, any, stream) : launch_down16_parity<IO, 5, 1, false>(p, any, stream);
        return rot ? launch_down16_parity<IO, 7, 1, true>(p, any, stream) : launch_down16_parity<IO, 7, 1, false>(p, any, stream);
    }
    if (K == 3) return launch_down16_parity<IO, 3, 2, false>(p, any, stream);
    if (K == 5) return launch_down16_parity<IO, 5, 2, false>(p, any, stream);
    return launch_down16_parity<IO, 7, 2, false>(p, any, stream);
}

template int try_launch_fir_tiled16<half_t>(const half_t *, const half_t *, half_t *, const Geometry &, hipStream_t);
template int try_launch_fir_tiled16<bf16_t>(const bf16_t *, const bf16_t *, bf16_t *, const Geometry &, hipStream_t);

}  // namespace dwconv
