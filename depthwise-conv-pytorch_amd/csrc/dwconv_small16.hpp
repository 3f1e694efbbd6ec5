// 16-bit LDS images for the whole-plane kernels (dwconv_small_fir.hpp, dwconv_small_bwd.hpp): runs of planes travel into LDS and
// back as they are in memory, a lane's rows are dwords of two elements, and sums take two products at a time (two-element dot
// products: each rounds like two multiply-adds of widened elements, subnormals kept; a product beyond fp32's range is an infinity).
//
// With fp32 images these kernels were bound by the instructions they issue: every element widened on its way in, K * K
// multiply-adds a result.  Pairs cost next to nothing here, because a lane holds whole rows:
//   * horizontally a pair of elements is a dword of the row as loaded.  A window of K (odd) elements is cut on even columns, so
//     it is made of K / 2 such dwords and one element at its left or right end, whichever parity its first column has;
//   * the elements left over pair up vertically: the same column of two rows is one byte permutation, shared by every result
//     that needs it.  Only a window's last element, of K * K, is a multiply-add of a widened one.
// us before / after (fp32 images / these): both gradients, bf16 batch 128, 28x28 C=240 5x5 58.5 / 48.9, 14x14 C=672 5x5 40.5 / 35.6,
// C=480 3x3 23.7 / 21.8; batch 64 19x19 C=672 5x5 64.6 / 57.4, 16x16 C=672 5x5 38.4 / 24.8; forward, 14x14 C=672 5x5 stride 2
// 13.5 / 10.9, fp16 28x28 C=240 5x5 31.2 / 23.7, bf16 batch 64 32x32 C=240 5x5 30.1 / 15.5 (its fp32 rows meet on the same banks).  Of
// the 29 us of 14x14 C=480 5x5 both gradients 13 are launches, first loads and the sums' way out, 13 the products, 4 memory.
// No product is made for the sake of a pair (no zero taps, no zero elements), so in the forward pass and in grad-input an infinity
// reaches the results of its windows only.  Grad-weight multiplies the padding's zeros, as with fp32 images: those of the rows above
// and below a plane and of a lane's rows past it, and in the ragged instances those of the columns past a row.  An infinity
// that they meet makes NaN of taps it has no part in.
#pragma once

#include "dwconv_small_common.hpp"
#include "dwconv_tile16_common.hpp"

namespace dwconv {

namespace {

// dwords of a row of n elements
constexpr int row_dwords(int n) { return (n + 1) / 2; }

// The low (h = 0) or high element of a dword as fp32.
template <typename IO>
__device__ __forceinline__ float widen_half(uint32_t d, int h)
{
    if constexpr (std::is_same<IO, bf16_t>::value) return __uint_as_float(h ? d & 0xffff0000u : d << 16);
    else return Io<IO>::in(__builtin_bit_cast(IO, static_cast<uint16_t>(h ? d >> 16 : d & 0xffffu)));
}
// low or high elements of two dwords: a in the low half, b in the high one
__device__ __forceinline__ uint32_t pair_of_halves(uint32_t a, uint32_t b, int h)
{
    return __builtin_amdgcn_perm(b, a, h ? 0x07060302u : 0x05040100u);
}

// A row of N elements (RAG: of w <= N, zeros from there on) that starts at element `at` of the 16-bit image, as dwords.  Exact
// even widths: rows start on even elements, on multiples of four or eight if N is one.  Every other width: on any element, and
// the dwords are shifted into place.
template <int N, bool RAG>
__device__ __forceinline__ void lds_load_row16(const uint16_t *image, int at, uint32_t (&d)[row_dwords(N)], int w)
{
    constexpr int ND = row_dwords(N);
    if constexpr (!RAG && N % 2 == 0) {
        const uint16_t *p = image + at;
        if constexpr (N % 8 == 0) {
#pragma unroll
            for (int i = 0; i < ND / 4; ++i) {
                const u32x4 v = reinterpret_cast<const u32x4 *>(p)[i];
                d[4 * i] = v.x, d[4 * i + 1] = v.y, d[4 * i + 2] = v.z, d[4 * i + 3] = v.w;
            }
        } else if constexpr (N % 4 == 0) {
#pragma unroll
            for (int i = 0; i < ND / 2; ++i) {
                const u32x2 v = reinterpret_cast<const u32x2 *>(p)[i];
                d[2 * i] = v.x, d[2 * i + 1] = v.y;
            }
        } else {
#pragma unroll
            for (int i = 0; i < ND; ++i) d[i] = reinterpret_cast<const uint32_t *>(p)[i];
        }
    } else {
        const uint32_t *p = reinterpret_cast<const uint32_t *>(image) + (at >> 1);
        const unsigned sh = (at & 1) << 4;
        uint32_t raw[ND + 1];
#pragma unroll
        for (int i = 0; i < ND; ++i) raw[i] = p[i];
        raw[ND] = N % 2 == 0 ? p[ND] : 0u;  // (an odd row ends inside its ND dwords either way)
#pragma unroll
        for (int i = 0; i < ND; ++i) d[i] = __builtin_amdgcn_alignbit(raw[i + 1], raw[i], sh);
        if constexpr (RAG) {
            // (a capacity class spans eight widths)
#pragma unroll
            for (int i = (N > 7 ? (N - 7) / 2 : 0); i < ND; ++i) d[i] &= w > 2 * i + 1 ? ~0u : (w > 2 * i ? 0xffffu : 0u);
        } else {
            d[ND - 1] &= 0xffffu;
        }
    }
}

// A row of results.
template <typename IO, int N, bool RAG>
__device__ __forceinline__ void lds_store_row16(uint16_t *image, int at, const float *r, int w)
{
    constexpr int ND = row_dwords(N);
    uint32_t d[ND];
#pragma unroll
    for (int i = 0; i < ND; ++i) {
        const float a = r[2 * i], b = 2 * i + 1 < N ? r[2 * i + 1 < N ? 2 * i + 1 : 0] : 0.f;
        if constexpr (std::is_same<IO, bf16_t>::value) d[i] = bf16_pack2(a, b);
        else d[i] = f16_pack2(a, b);
    }
    if constexpr (!RAG && N % 2 == 0) {
        uint16_t *p = image + at;
        if constexpr (N % 4 == 0) {
#pragma unroll
            for (int i = 0; i < ND / 2; ++i) reinterpret_cast<uint2 *>(p)[i] = make_uint2(d[2 * i], d[2 * i + 1]);
        } else {
#pragma unroll
            for (int i = 0; i < ND; ++i) reinterpret_cast<uint32_t *>(p)[i] = d[i];
        }
    } else {
        lds_put_run16(image, at, RAG ? w : N, d);
    }
}

// Flat runs, as run_to_lds and lds_to_run but without a change of format.
template <typename IO>
__device__ __forceinline__ void run_to_lds16(const IO *__restrict__ g, uint16_t *lds, int n)
{
    const int n4 = n >> 2;
    for (int base = threadIdx.x; base < n4; base += kWave * kRunBatch) {
        uint2 v[kRunBatch];
#pragma unroll
        for (int u = 0; u < kRunBatch; ++u) v[u] = load4_raw<IO>(g + 4 * min(base + u * kWave, n4 - 1));
#pragma unroll
        for (int u = 0; u < kRunBatch; ++u) reinterpret_cast<uint2 *>(lds)[min(base + u * kWave, n4 - 1)] = v[u];
    }
    const int tail = n4 * 4 + threadIdx.x;
    if (tail < n) lds[tail] = reinterpret_cast<const uint16_t *>(g)[tail];
}
template <typename IO>
__device__ __forceinline__ void lds_to_run16(IO *__restrict__ g, const uint16_t *lds, int n, int head)
{
    const int n4 = n >> 2;
    constexpr int U = 4;
    const __amdgpu_buffer_rsrc_t view = buffer_view(g, static_cast<long>(n) * 2);
    for (int base = threadIdx.x; base < n4; base += kWave * U) {
        u32x2 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = reinterpret_cast<const u32x2 *>(lds)[min(base + u * kWave, n4 - 1)];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = base + u * kWave;
            const bool whole = i < n4 && (i > 0 || head == 0);
            __builtin_amdgcn_raw_buffer_store_b64(v[u], view, whole ? i * 8u : kOob, 0, kStoreStreaming);
        }
    }
    const int t = threadIdx.x;
    uint16_t *const to = reinterpret_cast<uint16_t *>(g);
    if (head != 0 && n4 > 0 && t >= head && t < 4) to[t] = lds[t];
    const int tail = n4 * 4 + t;
    if (tail < n && tail >= head) to[tail] = lds[tail];
}
// Channel of the lane's plane (plane0: uniform).  Divided in 32 bits where they do: the 64-bit remainder is some hundred
// instructions in front of everything else.
__device__ __forceinline__ int plane_channel(long plane0, int pl, long planes, int channels)
{
    if (planes < (1l << 31)) {
        const unsigned first = static_cast<unsigned>(plane0) % static_cast<unsigned>(channels);
        return static_cast<int>((first + pl) % static_cast<unsigned>(channels));
    }
    return static_cast<int>((plane0 + pl) % channels);
}

// zeros of the row that stands in for those above and below a plane: from element `at` (a multiple of eight) on
template <int W>
__device__ __forceinline__ void clear_zero_row16(uint16_t *image, int at)
{
    if (threadIdx.x < W / 8 + 2) reinterpret_cast<uint4 *>(image + at)[threadIdx.x] = make_uint4(0u, 0u, 0u, 0u);
}
constexpr int zero_row_elems16(int w) { return (w / 8 + 2) * 8; }

// A channel's taps as horizontal pairs (tx, tx + 1), vertical pairs (ty, ty + 1) and fp32.  What a kernel does not use it does
// not compute.  They are read 16 bytes at a time from the 32-bit boundary before the channel's first one (a load per tap was
// more loads than the lane's share of the planes), through a view of the whole filter tensor.
template <typename IO, int K>
struct Taps16 {
    uint32_t h[K][K - 1], v[K - 1][K];
    float f[K][K];
    template <bool FLIP>
    __device__ __forceinline__ void load(const void *taps, int c, int channels)
    {
        constexpr int KK = K * K, ND = row_dwords(KK), NQ = (ND + 1 + 3) / 4;
        const AnyWidthView view = any_width_view(static_cast<const IO *>(taps), static_cast<long>(channels) * KK * 2);
        const unsigned at = static_cast<unsigned>(c) * (KK * 2u) + view.bias, sh = (at & 2u) << 3;
        uint32_t raw[4 * NQ], e[ND];
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const u32x4 t = __builtin_amdgcn_raw_buffer_load_b128(view.view, (at & ~3u) + 16u * q, 0, 0);
            raw[4 * q] = t.x, raw[4 * q + 1] = t.y, raw[4 * q + 2] = t.z, raw[4 * q + 3] = t.w;
        }
#pragma unroll
        for (int i = 0; i < ND; ++i) e[i] = __builtin_amdgcn_alignbit(raw[i + 1], raw[i], sh);
        auto index = [](int y, int x) { return FLIP ? KK - 1 - (y * K + x) : y * K + x; };
        auto pair = [&](int a, int b) {
            return __builtin_amdgcn_perm(e[b / 2], e[a / 2], (a & 1 ? 0x0302u : 0x0100u) | (b & 1 ? 0x07060000u : 0x05040000u));
        };
#pragma unroll
        for (int y = 0; y < K; ++y)
#pragma unroll
            for (int x = 0; x < K; ++x) {
                f[y][x] = widen_half<IO>(e[index(y, x) / 2], index(y, x) & 1);
                if (x + 1 < K) h[y][x] = pair(index(y, x), index(y, x + 1));
                if (y + 1 < K) v[y][x] = pair(index(y, x), index(y + 1, x));
            }
    }
};

// How the window of result o (columns o * S - K/2 + tx of a row of W) is cut.
template <int W, int K, int S>
struct Cut16 {
    static constexpr int col(int o, int tx) { return o * S - K / 2 + tx; }
    static constexpr bool inside(int o, int tx) { return col(o, tx) >= 0 && col(o, tx) < W; }
    static constexpr bool starts_pair(int o, int tx)
    {
        return tx + 1 < K && inside(o, tx) && (col(o, tx) & 1) == 0 && col(o, tx) + 1 < W;
    }
    static constexpr bool single(int o, int tx)
    {
        return inside(o, tx) && !starts_pair(o, tx) && !(tx > 0 && starts_pair(o, tx > 0 ? tx - 1 : 0));
    }
};

// sum[b][o] += window of result row b, column o: window rows come from load(wr, dwords), one ahead of their use.
template <typename IO, int W, int K, int S, int BH, int OW, typename LOAD>
__device__ __forceinline__ void convolve16(const Taps16<IO, K> &t, LOAD load, float (&sum)[BH][OW])
{
    using C = Cut16<W, K, S>;
    constexpr int ND = row_dwords(W), ROWS = (BH - 1) * S + K;
    uint32_t rows[3][ND];  // the previous row, this one and the next
    load(0, rows[0]);
#pragma unroll
    for (int wr = 0; wr < ROWS; ++wr) {
        const uint32_t(&d)[ND] = rows[wr % 3];
        const uint32_t(&before)[ND] = rows[(wr + 2) % 3];
        if (wr + 1 < ROWS) load(wr + 1, rows[(wr + 1) % 3]);
        uint32_t vp[W];  // columns of rows wr - 1 and wr (odd wr)
        float one[W];
#pragma unroll
        for (int i = 0; i < W; ++i) {
            if (wr & 1) vp[i] = pair_of_halves(before[i / 2], d[i / 2], i & 1);
            one[i] = widen_half<IO>(d[i / 2], i & 1);
        }
#pragma unroll
        for (int b = 0; b < BH; ++b) {
            const int ty = wr - b * S;
            if (ty < 0 || ty >= K) continue;
            // rows pair up on even window rows: the row left over is a result's last one, or its first where that is odd
            const bool second = (wr & 1) != 0 && ty > 0;
            const bool alone = (wr & 1) != 0 ? ty == 0 : ty == K - 1;
#pragma unroll
            for (int o = 0; o < OW; ++o) {
#pragma unroll
                for (int tx = 0; tx < K; ++tx) {
                    const int ix = C::col(o, tx);
                    if (C::starts_pair(o, tx)) {
                        sum[b][o] = dot2<IO>(d[ix / 2], t.h[ty][tx < K - 1 ? tx : 0], sum[b][o]);
                    } else if (C::single(o, tx)) {
                        if (second) sum[b][o] = dot2<IO>(vp[ix], t.v[ty > 0 ? ty - 1 : 0][tx], sum[b][o]);
                        else if (alone) sum[b][o] = fmaf(one[ix], t.f[ty][tx], sum[b][o]);
                    }
                }
            }
        }
        pin_registers(sum);
    }
}

// sum[ty * K + tx] += the lane's BH rows of out_grad (g, dwords of OW elements) against the rows of x they meet, stride 1.
template <typename IO, int W, int K, int BH, typename LOAD>
__device__ __forceinline__ void grad_weight16(const uint32_t (&g)[BH][row_dwords(W)], LOAD load, float (&sum)[K * K])
{
    constexpr int ND = row_dwords(W), P = K / 2, ROWS = BH - 1 + K;
    uint32_t rows[2][ND];
    load(0, rows[0]);
#pragma unroll
    for (int wr = 0; wr < ROWS; ++wr) {
        const uint32_t(&d)[ND] = rows[wr & 1];
        if (wr + 1 < ROWS) load(wr + 1, rows[(wr + 1) & 1]);
        uint32_t odd[ND];  // elements 2 i + 1 and 2 i + 2
#pragma unroll
        for (int i = 0; i + 1 < ND; ++i) odd[i] = __builtin_amdgcn_alignbit(d[i + 1], d[i], 16);
#pragma unroll
        for (int b = 0; b < BH; ++b) {
            const int ty = wr - b;
            if (ty < 0 || ty >= K) continue;
#pragma unroll
            for (int tx = 0; tx < K; ++tx)
#pragma unroll
                for (int o = 0; o < W; o += 2) {
                    const int ix = o - P + tx;
                    const bool first = ix >= 0 && ix < W, second = o + 1 < W && ix + 1 >= 0 && ix + 1 < W;
                    float &s = sum[ty * K + tx];
                    if (first && second) s = dot2<IO>(g[b][o / 2], (ix & 1) ? odd[ix / 2] : d[ix / 2], s);
                    else if (first) s = fmaf(widen_half<IO>(g[b][o / 2], 0), widen_half<IO>(d[ix / 2], ix & 1), s);
                    else if (second) s = fmaf(widen_half<IO>(g[b][o / 2], 1), widen_half<IO>(d[(ix + 1) / 2], (ix + 1) & 1), s);
                }
        }
        pin_registers(sum);
    }
}

}  // namespace

}  // namespace dwconv
