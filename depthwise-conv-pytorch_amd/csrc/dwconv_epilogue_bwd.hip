// Backward of the fused forward epilogue  out = act(conv * scale[c] + shift[c])  (dwconv2d_fused_*).
//
// Given the convolution result `conv` (recomputed by the caller with the plain forward kernel; the fused
// forward keeps nothing but its inputs) and the gradient of `out`, one sweep produces
//   conv_grad  = out_grad * act'(z) * scale[c],          z = conv * scale[c] + shift[c]
//   scale_grad[c] = sum_{n,y,x} out_grad * act'(z) * conv
//   shift_grad[c] = sum_{n,y,x} out_grad * act'(z)
// conv_grad then goes through the ordinary backward kernels as out_grad.  Three tensor sweeps (two reads, one
// write) stand for the four elementwise backward passes autograd would run for mul, add and the activation.
// The per-channel sums are two-pass and bit-identical from run to run: partial[c][chunk][2] per workgroup
// (fixed-order tree in LDS), then the fixed-order fp64 sum shared with grad-weight.
// No counterpart in the reference, which has no epilogue (it rejects a bias, torch_dwconv/dwconv.py:108-109).
#include "dwconv_tile_common.hpp"

#include <algorithm>

namespace dwconv {

namespace {

constexpr int kEpiThreads = 256;

struct EpiBwdPlan {
    const void *conv;
    const void *out_grad;
    void *conv_grad;
    const float *scale;
    const float *shift;
    float *partial;
    int act;
    int channel;
    int outer;            // NCHW: images; channels-last: pixels of all images
    int inner;            // NCHW: elements per plane; channels-last: 1
    int chunks;
    int outer_per_chunk;
    int vec;              // groups of four elements may be moved with one access
    // channels-last
    int lanes;            // lanes that one pixel takes in a workgroup
    unsigned lanes_magic; // lane / lanes
    int pixels;           // pixels that a workgroup takes at a time
    int half;             // the largest power of two below pixels: the first step of the sum over them
};

// out_grad * d act(z) / dz.
__device__ __forceinline__ float act_backward(float z, float g, int act)
{
    if (act == DWCONV_ACT_RELU) return EpilogueBackward::slope<DWCONV_ACT_RELU>(z, g);
    if (act == DWCONV_ACT_RELU6) return EpilogueBackward::slope<DWCONV_ACT_RELU6>(z, g);
    if (act == DWCONV_ACT_SILU) return EpilogueBackward::slope<DWCONV_ACT_SILU>(z, g);
    return g;
}

// One element: returns conv_grad and adds to the two channel sums.
__device__ __forceinline__ float epi_element(float y, float g, float sc, float sh, int act, float &s_scale, float &s_shift)
{
    const float ga = act_backward(fmaf(y, sc, sh), g, act);
    s_scale = fmaf(ga, y, s_scale);
    s_shift += ga;
    return ga * sc;
}

// CV consecutive elements as fp32, and conv_grad of them in their place.
template <typename IO, int CV>
__device__ __forceinline__ void epi_load(const IO *from, float (&v)[CV])
{
    if constexpr (CV == 4) {
        const float4 q = load4<IO>(from);
        v[0] = q.x, v[1] = q.y, v[2] = q.z, v[3] = q.w;
    } else {
        v[0] = Io<IO>::in(*from);
    }
}
template <typename IO, int CV>
__device__ __forceinline__ void epi_store(IO *to, const float (&v)[CV])
{
    if constexpr (CV == 4) store4<IO>(to, v[0], v[1], v[2], v[3]);
    else *to = Io<IO>::out(v[0]);
}

// Rows of pixels that the end of the channels-last kernel adds in one go, and that a long chunk is a multiple of.
constexpr int kEpiRows = 4;

// Sum of v over the workgroup, in a fixed order, valid in lane 0.
__device__ __forceinline__ float block_sum(float v, float *red)
{
    red[threadIdx.x] = v;
    __syncthreads();
#pragma unroll
    for (int half = kEpiThreads / 2; half > 0; half >>= 1) {
        if (static_cast<int>(threadIdx.x) < half) red[threadIdx.x] += red[threadIdx.x + half];
        __syncthreads();
    }
    const float s = red[0];
    __syncthreads();
    return s;
}

// NCHW: workgroup (channel c, chunk of images); lanes run along the plane.
template <typename IO>
__global__ __launch_bounds__(kEpiThreads) void epilogue_bwd_nchw_kernel(const EpiBwdPlan p)
{
    __shared__ float red[kEpiThreads];
    const int c = blockIdx.x, chunk = blockIdx.y;
    const int n0 = chunk * p.outer_per_chunk, n1 = min(p.outer, n0 + p.outer_per_chunk);
    const float sc = p.scale != nullptr ? p.scale[c] : 1.f, sh = p.shift != nullptr ? p.shift[c] : 0.f;
    const IO *const conv = static_cast<const IO *>(p.conv);
    const IO *const gy = static_cast<const IO *>(p.out_grad);
    IO *const g0 = static_cast<IO *>(p.conv_grad);
    float s_scale = 0.f, s_shift = 0.f;
    if (p.vec) {
        const int inner4 = p.inner >> 2;
        const int total = (n1 - n0) * inner4;
        for (int e = threadIdx.x; e < total; e += kEpiThreads) {
            const int n = e / inner4, i = e - n * inner4;
            const long off = (static_cast<long>(n0 + n) * p.channel + c) * p.inner + 4 * i;
            const float4 y = load4<IO>(conv + off), g = load4<IO>(gy + off);
            store4<IO>(g0 + off, epi_element(y.x, g.x, sc, sh, p.act, s_scale, s_shift),
                       epi_element(y.y, g.y, sc, sh, p.act, s_scale, s_shift),
                       epi_element(y.z, g.z, sc, sh, p.act, s_scale, s_shift),
                       epi_element(y.w, g.w, sc, sh, p.act, s_scale, s_shift));
        }
    } else {
        const int total = (n1 - n0) * p.inner;
        for (int e = threadIdx.x; e < total; e += kEpiThreads) {
            const int n = e / p.inner, i = e - n * p.inner;
            const long off = (static_cast<long>(n0 + n) * p.channel + c) * p.inner + i;
            g0[off] = Io<IO>::out(epi_element(Io<IO>::in(conv[off]), Io<IO>::in(gy[off]), sc, sh, p.act, s_scale, s_shift));
        }
    }
    const float t_scale = block_sum(s_scale, red), t_shift = block_sum(s_shift, red);
    if (threadIdx.x == 0) {
        float *dst = p.partial + (static_cast<long>(c) * p.chunks + chunk) * 2;
        dst[0] = t_scale;
        dst[1] = t_shift;
    }
}

// Channels-last: workgroup (p.lanes lanes of CV channels each, chunk of pixels).  The sweep is bound by HBM when every
// lane has work: with a wavefront per pixel whatever the channel count, 32 channels kept 8 lanes of 64 busy.  So a
// workgroup takes 256 / p.lanes pixels at a time, consecutive lanes consecutive addresses across pixels as well.  A lane
// has B pixels of both tensors in flight (conv_grad may lie over conv, so the compiler moves no load across a store): 32
// bytes of each, more is code that a small pass fetches and runs once (batch 64, C=768, 7x7, fp32: B=4 13.6 us, 2 12.5;
// batch 128, C=672, 14x14: 52.1 / 51.7, bf16 31.4 / 32.5).  Small passes are bound by latency, of the sum at the end too:
// the rows of lanes that share channels are halved in LDS down to kEpiRows, which all lanes then add, channel by channel.
// us, SiLU, a wavefront per pixel / this (TB/s of the three sweeps):
//   batch 128  C=32 112x112 fp32 312 / 142 (4.4), bf16 344 / 85 (3.6)   C=96 56x56 119 / 113 (4.1), bf16 102 / 71 (3.3)
//              C=144 56x56 167 / 163 (4.3), bf16 108 / 96 (3.6)         C=240 14x14 31.6 / 31.0, bf16 28.8 / 28.0
//              C=672 14x14 55.1 / 52.6, bf16 32.5 / 31.5                C=1152 7x7 25.8 / 25.5, bf16 21.0 / 20.3
//   batch 8    C=4 14x14 8.1 / 6.8    C=32 56x56 22 / 9.2   C=240 28x28 12.4 / 12.4, bf16 11.7 / 12.0   C=1152 7x7 7.6 / 7.6
template <typename IO, int CV>
__global__ __launch_bounds__(kEpiThreads) void epilogue_bwd_nhwc_kernel(const EpiBwdPlan p)
{
    constexpr int B = CV == 1 ? 1 : 8 / sizeof(IO);
    __shared__ float red[2 * CV][kEpiThreads];
    const int pl = fast_div(threadIdx.x, p.lanes_magic), cl = threadIdx.x - pl * p.lanes;
    const int c0 = (blockIdx.x * p.lanes + cl) * CV;
    const int chunk = blockIdx.y;
    const int o0 = chunk * p.outer_per_chunk, o1 = o0 + min(p.outer - o0, p.outer_per_chunk);  // o0 + a chunk may pass 2^31
    const bool live = pl < p.pixels && c0 < p.channel;
    const IO *const conv = static_cast<const IO *>(p.conv);
    const IO *const gy = static_cast<const IO *>(p.out_grad);
    IO *const g0 = static_cast<IO *>(p.conv_grad);
    float sc[CV], sh[CV], s_scale[CV], s_shift[CV];
#pragma unroll
    for (int v = 0; v < CV; ++v) {
        sc[v] = live && p.scale != nullptr ? p.scale[c0 + v] : 1.f;
        sh[v] = live && p.shift != nullptr ? p.shift[c0 + v] : 0.f;
        s_scale[v] = s_shift[v] = 0.f;
    }
    if (live) {
        const long step = static_cast<long>(p.pixels) * p.channel;
        long off = static_cast<long>(o0 + pl) * p.channel + c0;
        for (int left = o1 - o0 - pl; left > 0; left -= B * p.pixels, off += B * step) {
            float y[B][CV], g[B][CV];
            if ((B - 1) * p.pixels < left) {
#pragma unroll
                for (int u = 0; u < B; ++u) {
                    epi_load<IO, CV>(conv + off + u * step, y[u]);
                    epi_load<IO, CV>(gy + off + u * step, g[u]);
                }
            } else {
#pragma unroll
                for (int u = 0; u < B - 1; ++u) {
                    if (u * p.pixels >= left) break;
                    epi_load<IO, CV>(conv + off + u * step, y[u]);
                    epi_load<IO, CV>(gy + off + u * step, g[u]);
                }
            }
#pragma unroll
            for (int u = 0; u < B; ++u) {
                if (u * p.pixels >= left) break;
                float out[CV];
#pragma unroll
                for (int v = 0; v < CV; ++v) out[v] = epi_element(y[u][v], g[u][v], sc[v], sh[v], p.act, s_scale[v], s_shift[v]);
                epi_store<IO, CV>(g0 + off + u * step, out);
            }
        }
    }
#pragma unroll
    for (int v = 0; v < CV; ++v) {
        red[2 * v][threadIdx.x] = s_scale[v];
        red[2 * v + 1][threadIdx.x] = s_shift[v];
    }
    __syncthreads();
    int rows = p.pixels;
    for (int half = p.half; half >= kEpiRows; half >>= 1) {
        if (pl < half && pl + half < rows) {
#pragma unroll
            for (int v = 0; v < 2 * CV; ++v) red[v][threadIdx.x] += red[v][threadIdx.x + half * p.lanes];
        }
        rows = half;
        __syncthreads();
    }
    for (int i = threadIdx.x; i < CV * p.lanes; i += kEpiThreads) {
        const int v = fast_div(i, p.lanes_magic), lane = i - v * p.lanes, c = (blockIdx.x * p.lanes + lane) * CV + v;
        float a[kEpiRows], b[kEpiRows];
#pragma unroll
        for (int r = 0; r < kEpiRows; ++r) {
            const int at = min(r, rows - 1) * p.lanes + lane;
            a[r] = red[2 * v][at];
            b[r] = red[2 * v + 1][at];
        }
#pragma unroll
        for (int r = 1; r < kEpiRows; ++r) {
            a[0] += r < rows ? a[r] : 0.f;
            b[0] += r < rows ? b[r] : 0.f;
        }
        if (c < p.channel) {
            float *dst = p.partial + (static_cast<long>(c) * p.chunks + chunk) * 2;
            dst[0] = a[0];
            dst[1] = b[0];
        }
    }
}

// Lanes for `groups` channel groups: all of them where a wavefront holds them, else equal shares of whole eights of lanes
// (a 128-byte line where a lane moves four fp32 channels).
int lanes_for(int groups)
{
    const int blocks = ceil_div(groups, 64), share = ceil_div(groups, blocks);
    return blocks == 1 ? share : (share + 7) / 8 * 8;
}

bool make_plan(EpiBwdPlan &p, int batch, int channel, int out_h, int out_w, bool channels_last)
{
    const long plane = static_cast<long>(out_h) * out_w;
    p.channel = channel;
    if (channels_last) {
        if (batch * plane >= (1l << 31)) return false;
        p.outer = static_cast<int>(batch * plane);
        p.inner = 1;
        const int groups = ceil_div(channel, 64 * (channel % 4 == 0 ? 4 : 1));
        int chunks = ceil_div(2048, groups);
        chunks = std::max(1, std::min(chunks, std::min(ceil_div(p.outer, 16), 65535)));
        p.outer_per_chunk = ceil_div(p.outer, chunks);
        // A chunk takes the pixels that a workgroup works on at a time, or whole multiples of them, and up to kEpiRows times
        // as many where that leaves 128 chunks or more: partial sums are the larger part of a small pass (batch 8, fp32,
        // C=8 56x56: chunks of 16 pixels 26.7 us, of a workgroup's 128 and more 7.3).  Longer chunks are whole batches of four
        // (batch 128, 28x28, C=80 bf16: multiples of one 28.7, of four 24.9; batch 100, 50x50, C=36 30.0 / 25.8), except
        // where lanes hold single elements and the workgroups' balance counts for more (128x255x14x14 bf16 21.2 / 24.0).
        const bool quads = channel % 4 == 0;
        const int pixels = kEpiThreads / lanes_for(quads ? channel / 4 : channel), batch_pixels = kEpiRows * pixels;
        p.outer_per_chunk = std::max(p.outer_per_chunk, std::min(batch_pixels, ceil_div(p.outer, 128)));
        const int unit = quads && p.outer_per_chunk > batch_pixels ? batch_pixels : pixels;
        p.outer_per_chunk = ceil_div(p.outer_per_chunk, unit) * unit;
    } else {
        if (plane >= (1l << 30)) return false;
        p.outer = batch;
        p.inner = static_cast<int>(plane);
        int chunks = ceil_div(4096, std::max(channel, 1));
        chunks = std::max(1, std::min(chunks, std::min(batch, 65535)));
        p.outer_per_chunk = ceil_div(batch, chunks);
        // a chunk's elements of one channel are indexed with 32 bits
        while (static_cast<long>(p.outer_per_chunk) * plane >= (1l << 31)) p.outer_per_chunk = ceil_div(p.outer_per_chunk, 2);
        if (ceil_div(batch, p.outer_per_chunk) > 65535) return false;
    }
    p.chunks = static_cast<int>((static_cast<long>(p.outer) + p.outer_per_chunk - 1) / p.outer_per_chunk);  // the sum may pass 2^31
    return true;
}

}  // namespace

size_t epilogue_backward_workspace(int batch, int channel, int out_h, int out_w, bool channels_last)
{
    EpiBwdPlan p{};
    if (batch <= 0 || channel <= 0 || out_h <= 0 || out_w <= 0) return 0;
    if (!make_plan(p, batch, channel, out_h, out_w, channels_last)) return 0;
    return static_cast<size_t>(channel) * p.chunks * 2 * sizeof(float);
}

template <typename IO>
int epilogue_backward(const IO *conv, const IO *out_grad, const float *scale, const float *shift, IO *conv_grad,
                      float *param_grad, void *ws, size_t ws_bytes, int batch, int channel, int out_h, int out_w, int act,
                      bool channels_last, hipStream_t stream)
{
    EpiBwdPlan p{};
    if (!make_plan(p, batch, channel, out_h, out_w, channels_last)) return fail(DWCONV_ERR_UNSUPPORTED, "tensor too large");
    const size_t need = static_cast<size_t>(channel) * p.chunks * 2 * sizeof(float);
    if (ws == nullptr || ws_bytes < need)
        return fail(DWCONV_ERR_WORKSPACE, "the epilogue backward needs a workspace of %zu bytes, got %zu", need, ws_bytes);
    p.conv = conv;
    p.out_grad = out_grad;
    p.conv_grad = conv_grad;
    p.scale = scale;
    p.shift = shift;
    p.partial = static_cast<float *>(ws);
    p.act = act;
    const bool aligned = aligned4(conv) && aligned4(out_grad) && aligned4(conv_grad);
    if (channels_last) {
        p.vec = aligned && channel % 4 == 0;
        const int groups = p.vec ? channel / 4 : channel;
        p.lanes = lanes_for(groups);
        p.lanes_magic = magic_u16(static_cast<unsigned>(p.lanes));
        p.pixels = kEpiThreads / p.lanes;
        for (p.half = 1; 2 * p.half < p.pixels;) p.half *= 2;
        const dim3 grid(ceil_div(groups, p.lanes), p.chunks);
        if (p.vec) hipLaunchKernelGGL((epilogue_bwd_nhwc_kernel<IO, 4>), grid, dim3(kEpiThreads), 0, stream, p);
        else hipLaunchKernelGGL((epilogue_bwd_nhwc_kernel<IO, 1>), grid, dim3(kEpiThreads), 0, stream, p);
    } else {
        p.vec = aligned && p.inner % 4 == 0;
        hipLaunchKernelGGL(epilogue_bwd_nchw_kernel<IO>, dim3(channel, p.chunks), dim3(kEpiThreads), 0, stream, p);
    }
    const int rc = check_launch("epilogue_bwd_kernel");
    if (rc != DWCONV_OK) return rc;
    note_variant("epilogue_bwd%s<%s,v%d> chunks%d", sizeof(IO) == 2 ? "16" : "", channels_last ? "nhwc" : "nchw", p.vec ? 4 : 1,
                 p.chunks);
    // param_grad[c][0] = scale_grad, [c][1] = shift_grad: the fixed-order fp64 sum over the chunks
    return launch_wgrad_final<float>(p.partial, param_grad, channel, 2, p.chunks, stream);
}

#define DWCONV_INSTANTIATE(IO)                                                                                          \
    template int epilogue_backward<IO>(const IO *, const IO *, const float *, const float *, IO *, float *, void *, size_t, \
                                       int, int, int, int, int, bool, hipStream_t);
DWCONV_INSTANTIATE(float)
DWCONV_INSTANTIATE(half_t)
DWCONV_INSTANTIATE(bf16_t)
#undef DWCONV_INSTANTIATE

}  // namespace dwconv
