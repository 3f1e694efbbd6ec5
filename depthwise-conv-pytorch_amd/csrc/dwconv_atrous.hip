// Dilated 3x3 layers at stride 1 with "same" padding (pad == dilation), any dilation (make_plan says where): forward, and both gradients in one
// sweep over out_grad.
//
// What bounds them is how much is moved per useful byte: with rates of 6 to 18 on maps of 33 to 97 columns the zero
// padding is up to half of a padded image, so a kernel that materialises it in LDS (fir_any_kernel, wgrad_any_kernel)
// spends most of its staging and LDS traffic on zeros.  Here a plane is copied into LDS as it lies in memory, one linear
// stream of 16-byte loads whatever the row width, and the padding exists only as one zero cell.
//
// Work split: a lane owns a column of one residue class of rows, i.e. the linear positions q, q + W*DH, q + 2*W*DH, ... of
// the plane.  Lanes of a wavefront own consecutive q, so LDS reads and global accesses are consecutive too, across row
// ends as well, and a step further down the column reads three new values for nine multiply-adds (forward) or eighteen
// (backward).  A position past the plane is past its buffer view (loads give zero, stores are dropped) and its LDS
// address is clamped to the zero cell; columns outside the row take the zero cell through their lane's offset.
//
// Staging is what has to be hidden: a workgroup walks a few planes of one channel and keeps the next plane's loads in
// flight in registers while it works on the one in LDS (without that the forward pass took 45 us instead of 26 at
// 65x65).  Batch 16, 256 channels, us, the any-geometry kernels before / this one:
//   65x65 fp32, rate 6:  forward 44 / 26, backward 127 / 36      rate 18: forward 55 / 26, backward 148 / 37
//   97x97 fp32, rate 18: forward 129 / 73, backward 293 / 109    65x65 bf16, rate 6: forward 44 / 18, backward 138 / 27
// (the 65x65 fp32 pair moves 138 and 208 MB: 5.3 and 5.7 TB/s).
#include "dwconv_tile_common.hpp"

#include <algorithm>

namespace dwconv {
namespace {

constexpr int kMaxThreads = 512;
constexpr int kMaxWaves = kMaxThreads / 64;
constexpr int kAtrousLds = 64 * 1024;
// 16-byte lines of the next plane that a lane holds at most
constexpr int kMaxAhead = 8;
static_assert(kMaxAhead * kMaxThreads * 16 >= kAtrousLds, "every plane that make_plan takes is staged whole");

struct AtrousPlan {
    int batch, channel, h, w;
    int dh, dw;
    int splits;       // workgroups per channel
    int per_split;    // images a workgroup takes
    int chains;       // columns x residue classes of rows
    int steps;        // positions of the longest chain
    unsigned w_magic; // q / w
};

// One element of the raw LDS image as fp32.
template <typename IO>
__device__ __forceinline__ float lds_value(const char *lds, unsigned at)
{
    return Io<IO>::in(*reinterpret_cast<const IO *>(lds + at));
}
template <typename IO>
__device__ __forceinline__ float view_value(__amdgpu_buffer_rsrc_t view, unsigned at)
{
    if constexpr (sizeof(IO) == 4) return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(view, at, 0, 0));
    else return Io<IO>::in(__builtin_bit_cast(IO, __builtin_amdgcn_raw_buffer_load_b16(view, at, 0, 0)));
}
template <typename IO>
__device__ __forceinline__ void view_put(__amdgpu_buffer_rsrc_t view, unsigned at, float v)
{
    if constexpr (sizeof(IO) == 4) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), view, at, 0, kStoreStreaming);
    else __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(unsigned short, Io<IO>::out(v)), view, at, 0, kStoreStreaming);
}

// FUSED: `in` is out_grad, `x` the input; out gets grad-input (the rotated taps) and partial[c][split][9] the
// grad-weight sums.  Otherwise `in` is the input and out the result.
template <typename IO, bool FUSED, int AHEAD>
__global__ __launch_bounds__(kMaxThreads) void atrous_kernel(const AtrousPlan p, const IO *__restrict__ in,
                                                             const IO *__restrict__ x, const IO *__restrict__ taps,
                                                             IO *__restrict__ out, float *__restrict__ partial)
{
    extern __shared__ __align__(16) char lds[];
    constexpr unsigned E = sizeof(IO);
    const int c = blockIdx.x, split = blockIdx.y;
    const int n0 = split * p.per_split, n1 = min(p.batch, n0 + p.per_split);
    const unsigned plane = static_cast<unsigned>(p.h) * p.w;
    const unsigned plane_bytes = plane * E;
    const unsigned step = static_cast<unsigned>(p.dh) * p.w * E;

    float w[9];
#pragma unroll
    for (int t = 0; t < 9; ++t) w[t] = Io<IO>::in(taps[static_cast<long>(c) * 9 + (FUSED ? 8 - t : t)]);
    float total[FUSED ? 9 : 1] = {};

    // The 16-byte lines that hold a plane (its first and last one may hold a neighbour's bytes too: never used).  A lane
    // keeps AHEAD lines of the next plane in flight while it works on this one: AHEAD * blockDim.x covers the plane.
    u32x4 ahead[AHEAD];
    const auto fetch = [&](int n) {
        const IO *from = in + (static_cast<long>(n) * p.channel + c) * plane;
        const unsigned head = static_cast<unsigned>(reinterpret_cast<uintptr_t>(from) & 15);
        const __amdgpu_buffer_rsrc_t src = buffer_view(reinterpret_cast<const char *>(from) - head, (head + plane_bytes + 15) & ~15u);
#pragma unroll
        for (int k = 0; k < AHEAD; ++k)
            ahead[k] = __builtin_amdgcn_raw_buffer_load_b128(src, (threadIdx.x + k * blockDim.x) * 16, 0, 0);
    };
    fetch(n0);
    for (int n = n0; n < n1; ++n) {
        const long base = (static_cast<long>(n) * p.channel + c) * plane;
        const unsigned head = static_cast<unsigned>(reinterpret_cast<uintptr_t>(in + base) & 15);
        const unsigned lines = (head + plane_bytes + 15) / 16;
        const unsigned zero = head + plane_bytes;  // the zero cell: the element after the plane's last one
        __syncthreads();  // the previous plane's image is no longer read
        u32x4 *image = reinterpret_cast<u32x4 *>(lds);
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) {
            const unsigned i = threadIdx.x + k * blockDim.x;
            if (i < lines) image[i] = ahead[k];
        }
        if (threadIdx.x == (lines - 1) % blockDim.x) {  // who wrote the last line: its wavefront's LDS writes stay in order
            asm volatile("" ::: "memory");
            *reinterpret_cast<IO *>(lds + zero) = Io<IO>::out(0.f);
        }
        __syncthreads();
        if (n + 1 < n1) fetch(n + 1);
        const __amdgpu_buffer_rsrc_t outs = buffer_view(out + base, plane_bytes);
        const __amdgpu_buffer_rsrc_t xs = buffer_view(FUSED ? x + base : in, FUSED ? plane_bytes : 0);

        for (int q = threadIdx.x; q < p.chains; q += blockDim.x) {
            const int col = q - fast_div(q, p.w_magic) * p.w;
            // byte offsets of the left and right neighbour; outside the row: past every address, i.e. the zero cell
            const bool has_l = col >= p.dw, has_r = col + p.dw < p.w;
            const unsigned left = has_l ? 0u - p.dw * E : kOob, right = has_r ? p.dw * E : kOob;
            unsigned at = q * E;                       // within the plane
            float above = 0.f, here = 0.f;             // sums of the rows before and at this position
            float acc[FUSED ? 9 : 1] = {};
            float x_prev = 0.f, x_now[2] = {}, x_next[2] = {};
            if constexpr (FUSED) {
                x_now[0] = view_value<IO>(xs, at);
                x_now[1] = view_value<IO>(xs, at + step);
            }
            for (int s = 0; s < p.steps; s += 2) {
                if constexpr (FUSED) {
                    x_next[0] = view_value<IO>(xs, at + 2 * step);
                    x_next[1] = view_value<IO>(xs, at + 3 * step);
                }
                float v[2][3];
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const unsigned a = at + k * step + head;
                    v[k][0] = lds_value<IO>(lds, min(a + left, zero));
                    v[k][1] = lds_value<IO>(lds, min(a, zero));
                    v[k][2] = lds_value<IO>(lds, min(a + right, zero));
                }
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const float done = fmaf(w[6], v[k][0], fmaf(w[7], v[k][1], fmaf(w[8], v[k][2], above)));
                    above = fmaf(w[3], v[k][0], fmaf(w[4], v[k][1], fmaf(w[5], v[k][2], here)));
                    here = fmaf(w[0], v[k][0], fmaf(w[1], v[k][1], w[2] * v[k][2]));
                    // the row before this one is complete (before the first: an offset that is past the view)
                    view_put<IO>(outs, s + k > 0 ? at + k * step - step : kOob, done);
                    if constexpr (FUSED) {
                        const float x_after = k == 0 ? x_now[1] : x_next[0];
                        // Padding meets nothing, so that a value that is not finite stays out of the sums it has no part in:
                        // a position past the plane meets no input of the row before, the first row has none before it
                        // and the last one none after it.
                        const float x_before = at + k * step < plane_bytes ? x_prev : 0.f;
                        const bool has_after = at + (k + 1) * step < plane_bytes;
#pragma unroll
                        for (int j = 0; j < 3; ++j) {
                            // out_grad at column col + (j - 1) * dw meets input column col through tap column 2 - j
                            if (s + k > 0) acc[2 - j] = fmaf(x_before, v[k][j], acc[2 - j]);
                            acc[3 + 2 - j] = fmaf(x_now[k], v[k][j], acc[3 + 2 - j]);
                            acc[6 + 2 - j] = fmaf(x_after, has_after ? v[k][j] : 0.f, acc[6 + 2 - j]);
                        }
                        x_prev = x_now[k];
                    }
                }
                if constexpr (FUSED) {
                    x_now[0] = x_next[0];
                    x_now[1] = x_next[1];
                }
                at += 2 * step;
            }
            // p.steps positions were walked, rounded up to a pair: the row after the last one read is still open
            view_put<IO>(outs, at - step, above);
            if constexpr (FUSED) {
                // sums of a column outside the row are those of zeros, and not a number where x is not finite: left out
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    total[3 * i + 2] += has_l ? acc[3 * i + 2] : 0.f;
                    total[3 * i + 1] += acc[3 * i + 1];
                    total[3 * i] += has_r ? acc[3 * i] : 0.f;
                }
            }
        }
    }
    if constexpr (FUSED) {
        __syncthreads();
        float *sums = reinterpret_cast<float *>(lds);
        const int waves = blockDim.x / 64;
#pragma unroll
        for (int t = 0; t < 9; ++t) {
            const float s = wave_sum_to_last_lane(total[t]);
            if ((threadIdx.x & 63) == 63) sums[(threadIdx.x >> 6) * 9 + t] = s;
        }
        __syncthreads();
        if (threadIdx.x < 9) {
            float s = sums[threadIdx.x];
            for (int k = 1; k < waves; ++k) s += sums[k * 9 + threadIdx.x];
            partial[(static_cast<long>(c) * p.splits + split) * 9 + threadIdx.x] = s;
        }
    }
}

// fused: for the backward kernel.
bool make_plan(AtrousPlan &p, const GeneralGeometry &g, size_t esize, bool fused)
{
    if (g.multiplier != 1 || g.kernel_h != 3 || g.kernel_w != 3 || g.stride_h != 1 || g.stride_w != 1) return false;
    if (g.pad_h != g.dil_h || g.pad_w != g.dil_w || g.batch < 1 || g.channel < 1 || g.in_h < 1 || g.in_w < 1) return false;
    if (env_int("DWCONV_ATROUS", 1) == 0) return false;
    const long plane_bytes = 1l * g.in_h * g.in_w * static_cast<long>(esize);
    if (plane_bytes + 48 > kAtrousLds) return false;  // the plane's 16-byte lines and the zero cell
    // dilations beyond the map reach only zeros: any that large are alike
    p.batch = g.batch;
    p.channel = g.channel;
    p.h = g.in_h;
    p.w = g.in_w;
    p.dh = g.dil_h < g.in_h ? g.dil_h : g.in_h;
    p.dw = g.dil_w < g.in_w ? g.dil_w : g.in_w;
    p.chains = p.dh * p.w;
    p.steps = ceil_div(p.h, p.dh);
    p.w_magic = magic_u16(static_cast<unsigned>(p.w));
    // Workgroups per CU: two or three walk several planes each where a plane's image or chains fill the CU (backward, us,
    // 512 / 768 workgroups: 65x65 fp32 39 / 36, 97x97 bf16 67 / 58; 80x80 fp32 64 / 71, 97x97 fp32 109 / 120, 128x128 bf16
    // 136 / 157).  Small planes are bound by the latency of a step, so up to 16 wavefronts of them, 24 of one each, and
    // eight in the forward pass once their bytes count (forward and backward, us, three a CU / these: batch 128, C=960 7x7
    // rate 3 fp32 86 and 129 / 31 and 42, C=480 14x14 56 and 88 / 24 and 36; batch 64, C=256 33x33 rate 6 30 and 44 / 27
    // and 42; with 12 a CU, batch 171, C=164 39x39 rate 3 forward 68 / 76).
    const int lanes = std::min(round_up(p.chains, 64), kMaxThreads);
    int per_cu = plane_bytes > 24 * 1024 ? 2 : 3;
    if (plane_bytes <= 12 * 1024) {
        const int waves = lanes == 64 ? 24 : fused || plane_bytes <= 4 * 1024 ? 16 : 8;
        per_cu = std::max(per_cu, std::min(waves * 64 / lanes, static_cast<int>(2 * kAtrousLds / (plane_bytes + 48))));
    }
    // A chain is walked row by row and a plane is never split, so a long chain takes as long as it takes whatever else the
    // CU does.  The any-geometry kernels split planes into bands: better where too few columns are in flight for the rows
    // there are, and the less so the more of their staging is padding or rows that are not a multiple of four long.  us,
    // any-geometry / this, fp32, rates vertical x horizontal:
    //   forward   batch 16, C=64: 400x40 1x2 34 / 68, 1000x16 1x3 57 / 227, 80x80 1x2 14 / 18; batch 4, C=32 97x97 1x2 7.8 / 10
    //             but 65x130 1x3 25 / 18, 120x60 2x3 21 / 15, 200x60 3x3 32 / 23; batch 7, C=712 278x26 3x3 106 / 80
    //   backward  batch 16, C=64: 400x40 1x2 88 / 133; batch 1, C=52 639x14 3x6 20 / 27
    //             but 120x120 1x2 79 / 52; batch 3, C=778 555x8 3x3 155 / 96
    const int serial = p.steps * ceil_div(p.chains, kMaxThreads);
    if (serial > 48) {
        const float planes = 1.f * g.batch * g.channel / kCus, ragged = p.w % 4 != 0 ? 1.4f : 1.f;
        const float padded = (1.f + 2.f * p.dh / p.h) * (1.f + 2.f * p.dw / p.w);
        const float columns = std::min<float>(per_cu, planes) * std::min(p.chains, kMaxThreads) * padded * ragged;
        if (fused) {
            if (serial > 160 && columns < 110.f) return false;
        } else if (p.dh > 2) {
            if (serial > 64 && planes < 1.f && columns < 140.f) return false;
        } else if (columns < (p.dh == 2 ? 125.f : p.dw > 3 ? 200.f : 265.f)) return false;
    }
    const int want = std::max(1, env_int("DWCONV_ATROUS_WGS", per_cu * kCus));
    const int splits = ceil_div(want, g.channel);
    p.per_split = ceil_div(g.batch, splits < g.batch ? splits : g.batch);
    p.splits = ceil_div(g.batch, p.per_split);
    return p.splits <= 65535;
}

// Whole wavefronts of chains, spread evenly over as few rounds as kMaxThreads lanes allow.
int threads_for(const AtrousPlan &p)
{
    const int waves = ceil_div(p.chains, 64), most = std::clamp(env_int("DWCONV_ATROUS_WAVES", kMaxWaves), 1, kMaxWaves);
    return 64 * ceil_div(waves, ceil_div(waves, most));
}

size_t lds_for(const AtrousPlan &p, size_t esize)
{
    const size_t image = (static_cast<size_t>(p.h) * p.w * esize + 15 + 15) / 16 * 16 + 16;
    const size_t sums = kMaxThreads / 64 * 9 * sizeof(float);
    return image > sums ? image : sums;
}

template <typename IO, bool FUSED>
int launch(const AtrousPlan &p, const IO *in, const IO *x, const IO *taps, IO *out, float *partial, hipStream_t stream)
{
    const int lines = (p.h * p.w * static_cast<int>(sizeof(IO)) + 15 + 15) / 16;
    const int most = std::clamp(env_int("DWCONV_ATROUS_AHEAD", kMaxAhead), ceil_div(lines, kMaxThreads), kMaxAhead);
    // as many wavefronts as the chains keep busy, more where the plane's lines need them
    int threads = threads_for(p);
    while (threads * most < lines) threads += 64;
    const dim3 grid(p.channel, p.splits), block(threads);
    const size_t bytes = lds_for(p, sizeof(IO));
    if (lines <= 3 * threads) hipLaunchKernelGGL((atrous_kernel<IO, FUSED, 3>), grid, block, bytes, stream, p, in, x, taps, out, partial);
    else if (lines <= 5 * threads) hipLaunchKernelGGL((atrous_kernel<IO, FUSED, 5>), grid, block, bytes, stream, p, in, x, taps, out, partial);
    else hipLaunchKernelGGL((atrous_kernel<IO, FUSED, kMaxAhead>), grid, block, bytes, stream, p, in, x, taps, out, partial);
    return check_launch("atrous_kernel");
}

}  // namespace

size_t atrous_workspace(const GeneralGeometry &g, size_t esize)
{
    AtrousPlan p;
    return make_plan(p, g, esize, true) ? static_cast<size_t>(p.channel) * p.splits * 9 * sizeof(float) : 0;
}

template <typename IO>
int try_launch_atrous_forward(const IO *in, const IO *taps, IO *out, const GeneralGeometry &g, hipStream_t stream)
{
    AtrousPlan p;
    if (!make_plan(p, g, sizeof(IO), false)) return -1;
    note_variant("atrous%s<k3x3,d%dx%d,fwd> splits%d images%d", sizeof(IO) == 2 ? "16" : "", g.dil_h, g.dil_w, p.splits, p.per_split);
    return launch<IO, false>(p, in, in, taps, out, nullptr, stream);
}

template <typename IO>
int try_launch_atrous_backward(const IO *in, const IO *gy, const IO *taps, IO *gx, IO *gw, void *ws, size_t ws_bytes,
                               const GeneralGeometry &g, hipStream_t stream)
{
    AtrousPlan p;
    if (!make_plan(p, g, sizeof(IO), true)) return -1;
    const size_t need = static_cast<size_t>(p.channel) * p.splits * 9 * sizeof(float);
    if (ws == nullptr || ws_bytes < need)
        return fail(DWCONV_ERR_WORKSPACE, "grad-weight needs a workspace of %zu bytes, got %zu", need, ws_bytes);
    note_variant("atrous_bwd%s<k3x3,d%dx%d> splits%d images%d", sizeof(IO) == 2 ? "16" : "", g.dil_h, g.dil_w, p.splits, p.per_split);
    const int rc = launch<IO, true>(p, gy, in, taps, gx, static_cast<float *>(ws), stream);
    if (rc != DWCONV_OK) return rc;
    return launch_wgrad_final(static_cast<const float *>(ws), gw, p.channel, 9, p.splits, stream);
}

#define DWCONV_INSTANTIATE(IO)                                                                                                \
    template int try_launch_atrous_forward<IO>(const IO *, const IO *, IO *, const GeneralGeometry &, hipStream_t);           \
    template int try_launch_atrous_backward<IO>(const IO *, const IO *, const IO *, IO *, IO *, void *, size_t,               \
                                                const GeneralGeometry &, hipStream_t);
DWCONV_INSTANTIATE(float)
DWCONV_INSTANTIATE(half_t)
DWCONV_INSTANTIATE(bf16_t)
#undef DWCONV_INSTANTIATE

}  // namespace dwconv
