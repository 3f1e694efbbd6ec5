"""The one-sweep backward of act(conv(x, w) * scale + shift) (``_C.dwconv2d_fused_backward``) at the edges of its tiles:
planes of one row and one column, last bands of few rows, several planes a workgroup, rows of any width, odd extents at
stride 2, all activations."""
import pytest
import torch
from torch.nn import functional as F

from shapes import make_inputs, shape_id

pytestmark = pytest.mark.gpu

ACT = {None: lambda z: z, "relu": F.relu, "relu6": F.relu6, "silu": F.silu}

CASES = [
    # whole planes: exact and ragged widths, channels that do not fill a wavefront (several images a workgroup: below)
    ((3, 12, 7, 7, 3, 1, 1), "small_bwd"), ((2, 5, 14, 14, 5, 1, 2), "small_bwd"), ((2, 7, 11, 13, 3, 1, 1), "small_bwd"),
    ((1, 3, 31, 29, 5, 1, 2), "small_bwd"), ((2, 6, 32, 32, 3, 2, 1), "small_bwd"), ((3, 4, 15, 15, 5, 2, 2), "small_bwd"),
    ((2, 3, 4, 1, 3, 1, 1), "small_bwd"), ((2, 4, 22, 22, 5, 1, 2), "small_bwd"),
    # tiles, stride 1: one row, less than a block, one row more than a band, several planes, rows of any width
    ((1, 2, 1, 48, 3, 1, 1), "bwd_tile"), ((2, 3, 3, 50, 5, 1, 2), "bwd_tile"), ((2, 9, 40, 36, 3, 1, 1), "bwd_tile"),
    ((1, 5, 38, 38, 5, 1, 2), "bwd_tile"), ((2, 3, 61, 56, 3, 1, 1), "bwd_tile"), ((1, 2, 75, 75, 3, 1, 1), "bwd_tile"),
    ((1, 2, 64, 129, 5, 1, 2), "bwd_tile"), ((2, 2, 112, 112, 3, 1, 1), "bwd_tile"), ((1, 1, 9, 257, 3, 1, 1), "bwd_tile"),
    # tiles, stride 2: odd and even extents
    ((1, 2, 1, 50, 3, 2, 1), "bwd_tile_s2"), ((2, 3, 38, 38, 3, 2, 1), "bwd_tile_s2"), ((1, 2, 75, 75, 5, 2, 2), "bwd_tile_s2"),
    ((2, 2, 112, 112, 3, 2, 1), "bwd_tile_s2"), ((1, 3, 57, 64, 5, 2, 2), "bwd_tile_s2"), ((1, 2, 6, 150, 3, 2, 1), "bwd_tile_s2"),
    ((1, 2, 150, 33, 5, 2, 2), "bwd_tile_s2"),
]


def params(c, gpu):
    g = torch.Generator().manual_seed(11)
    return (1.0 + 0.3 * torch.randn(c, generator=g)).to(gpu), (0.3 * torch.randn(c, generator=g)).to(gpu)


def reference(x, w, gy, scale, shift, act, stride, pad):
    x, w, scale, shift = (t.detach().cpu().double().requires_grad_(True) for t in (x, w, scale, shift))
    z = F.conv2d(x, w, stride=stride, padding=pad, groups=x.shape[1]) * scale.view(1, -1, 1, 1) + shift.view(1, -1, 1, 1)
    return torch.autograd.grad(ACT[act](z), (x, w, scale, shift), gy.cpu().double())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: shape_id(c[0]))
def test_one_sweep(gpu, case, dtype):
    """SiLU, whose gradient has no corners.  Everything is fp32 until it is stored: |error| <= u |ref| + 2e-5 of the largest
    result (u: half a step of a 16-bit type; fp32 sums of up to 3e4 products of order one, 2^-24 each and random)."""
    from torch_dwconv import _C

    shape, family = case
    n, c, h, w, k, s, p = shape
    x, wt, gy = (t.to(dtype).to(gpu) for t in make_inputs(shape, seed=3))
    scale, shift = params(c, gpu)
    grads = _C.dwconv2d_fused_backward(x, gy, wt, scale, shift, "silu", s, s, p, p)
    variant = _C.last_variant()
    assert variant.startswith(family) and ",epi>" in variant, variant
    u = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for got, ref, rounded in zip(grads, reference(x, wt, gy, scale, shift, "silu", s, p), (True, True, False, False)):
        assert got.shape == ref.shape
        err = (got.cpu().double() - ref).abs()
        bound = (u if rounded else 0.0) * ref.abs() + 2e-5 * ref.abs().max()
        assert bool((err <= bound).all()), (variant, float(err.max()), float(ref.abs().max()))
    again = _C.dwconv2d_fused_backward(x, gy, wt, scale, shift, "silu", s, s, p, p)
    assert all(torch.equal(a, b) for a, b in zip(grads, again))


# Grids capped to one workgroup a channel group: every workgroup walks all images.
ONE_WORKGROUP = ("DWCONV_SMALL_WGRAD_WAVES", "DWCONV_EPI_WGS", "DWCONV_S2_WGS_K3", "DWCONV_WGRAD_WGS")


def cap_grids(monkeypatch):
    monkeypatch.setenv("DWCONV_TUNING", "1")
    for name in ONE_WORKGROUP:
        monkeypatch.setenv(name, "1")


@pytest.mark.parametrize("shape", [(96, 16, 28, 28, 5, 1, 2), (96, 16, 7, 7, 3, 1, 1), (96, 16, 14, 14, 5, 2, 2), (96, 16, 13, 13, 3, 1, 1),
                                   (96, 16, 56, 56, 3, 1, 1), (96, 16, 36, 36, 3, 1, 1), (192, 16, 56, 56, 3, 2, 1)], ids=shape_id)
def test_scale_and_shift_sums_over_many_images(gpu, monkeypatch, shape):
    """fp32 sums over up to 3e5 elements, every workgroup on all images.  With u = 2^-24 and random signs: sums of 16 elements are off
    by sqrt(17 / 6) u of their size, images are added up in fp64, the tree over the lanes adds sqrt(10 / 3) u and the convolution
    under scale's gradient sqrt(25 / 6) u: 3.3 u together, u / 2 more for the results.  One fp32 sum over all images would be off
    by sqrt(n / 6) u, 16 to 21 u for 1344 to 2688 elements a lane (7x7 and 13x13: 8 to 15).  The bound is 6 u."""
    from torch_dwconv import _C

    cap_grids(monkeypatch)
    n, c, h, w, k, s, p = shape
    x, wt, gy = (t.to(gpu) for t in make_inputs(shape, seed=13))
    scale, shift = params(c, gpu)
    grads = _C.dwconv2d_fused_backward(x, gy, wt, scale, shift, None, s, s, p, p)
    assert " chunks1" in _C.last_variant(), _C.last_variant()
    for got, ref in zip(grads[2:], reference(x, wt, gy, scale, shift, None, s, p)[2:]):
        error = float((got.cpu().double() - ref).norm() / ref.norm())
        assert error <= 6 * 2.0 ** -24, (_C.last_variant(), error)


def check_against_64_bits(gpu, shape, dtype, seed):
    """As test_one_sweep; returns the variant."""
    from torch_dwconv import _C

    n, c, h, w, k, s, p = shape
    x, wt, gy = (t.to(dtype).to(gpu) for t in make_inputs(shape, seed=seed))
    scale, shift = params(c, gpu)
    grads = _C.dwconv2d_fused_backward(x, gy, wt, scale, shift, "silu", s, s, p, p)
    assert grads is not None
    variant = _C.last_variant()
    u = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    for got, ref, rounded in zip(grads, reference(x, wt, gy, scale, shift, "silu", s, p), (True, True, False, False)):
        err = (got.cpu().double() - ref).abs()
        bound = (u if rounded else 0.0) * ref.abs() + 2e-5 * ref.abs().max()
        assert bool((err <= bound).all()), (variant, float(err.max()), float(ref.abs().max()))
    return variant


# (shape, family): whole planes on and off 4-element boundaries, with and without the prefetch of the next image;
# tiles whose in_grad leaves through LDS (fp32 3x3, 56 and 60 columns), rows of any width, two planes a workgroup, two bands
SEVERAL = [((7, 5, 7, 7, 3, 1, 1), "small_bwd"), ((5, 4, 14, 14, 5, 1, 2), "small_bwd"), ((5, 3, 13, 11, 5, 1, 2), "small_bwd"),
           ((5, 3, 28, 28, 5, 1, 2), "small_bwd"), ((5, 3, 28, 28, 3, 2, 1), "small_bwd"), ((5, 3, 15, 15, 5, 2, 2), "small_bwd"),
           ((5, 2, 56, 56, 3, 1, 1), "bwd_tile"), ((3, 2, 130, 60, 3, 1, 1), "bwd_tile"), ((5, 3, 38, 38, 5, 1, 2), "bwd_tile"),
           ((5, 5, 33, 35, 3, 1, 1), "bwd_tile"), ((3, 1, 75, 75, 3, 1, 1), "bwd_tile"), ((3, 2, 64, 129, 5, 1, 2), "bwd_tile"),
           ((5, 3, 38, 38, 3, 2, 1), "bwd_tile_s2"), ((3, 1, 75, 75, 5, 2, 2), "bwd_tile_s2"), ((3, 2, 112, 112, 3, 2, 1), "bwd_tile_s2"),
           ((5, 1, 47, 57, 5, 2, 2), "bwd_tile_s2")]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["f32", "bf16", "f16"])
@pytest.mark.parametrize("case", SEVERAL, ids=lambda c: shape_id(c[0]))
def test_several_tiles_a_workgroup(gpu, monkeypatch, case, dtype):
    """One workgroup a channel group, so that it walks every image and band: LDS whose gy was replaced in place is staged again, the
    next image is prefetched, sums and results leave between tiles."""
    shape, family = case
    cap_grids(monkeypatch)
    variant = check_against_64_bits(gpu, shape, dtype, seed=29)
    assert variant.startswith(family) and ",epi>" in variant and variant.split(" chunks")[1].split(" ")[0] == "1", variant
    assert shape[0] >= 3


# Layers of 4 Mi elements and more, on both sides of the rules that send some of them to three calls; the same planes with fewer
# elements always take one sweep.
@pytest.mark.parametrize("shape,dtype,one_sweep", [
    ((9, 144, 64, 64, 3, 1, 1), torch.bfloat16, False), ((10, 144, 56, 56, 3, 1, 1), torch.bfloat16, True),
    ((9, 144, 64, 64, 5, 1, 2), torch.float32, False), ((9, 144, 64, 64, 3, 1, 1), torch.float32, True),
    ((9, 144, 64, 64, 5, 1, 2), torch.bfloat16, False), ((3, 144, 112, 112, 5, 1, 2), torch.bfloat16, False),
    ((5, 144, 80, 80, 5, 1, 2), torch.bfloat16, True), ((21, 144, 38, 38, 3, 2, 1), torch.bfloat16, False),
    ((19, 144, 40, 40, 3, 2, 1), torch.bfloat16, True), ((8, 144, 64, 64, 5, 2, 2), torch.bfloat16, False),
    ((10, 144, 56, 56, 5, 2, 2), torch.bfloat16, True), ((8, 144, 64, 64, 5, 2, 2), torch.float32, True)],
    ids=lambda v: shape_id(v) if isinstance(v, tuple) else str(v).split(".")[-1])
def test_which_large_layers_take_one_sweep(gpu, shape, dtype, one_sweep):
    from torch_dwconv import _C

    n, c, h, w, k, s, p = shape
    assert n * c * h * w >= 4 << 20 and (n // 2) * c * h * w < 4 << 20
    x, wt, gy = (t.to(dtype).to(gpu) for t in make_inputs(shape, seed=31))
    grads = _C.dwconv2d_fused_backward(x, gy, wt, None, None, "silu", s, s, p, p)
    assert (grads is not None) == one_sweep
    assert _C.dwconv2d_fused_backward(x[:n // 2], gy[:n // 2], wt, None, None, "silu", s, s, p, p) is not None
    if one_sweep:
        check_against_64_bits(gpu, shape, dtype, seed=31)


@pytest.mark.parametrize("shape", [(2, 4, 14, 14, 3, 1, 1), (1, 3, 29, 28, 5, 1, 2), (2, 2, 56, 56, 3, 1, 1), (1, 2, 75, 75, 3, 1, 1),
                                   (1, 2, 56, 56, 5, 2, 2)], ids=shape_id)
def test_silu_slope_is_that_of_the_separate_sweep(gpu, shape):
    """A filter that is one at its centre and zero elsewhere: the convolution is the input's elements, in_grad the slopes, both without
    a rounding.  The sigmoid is the rounded quotient in both, so the bits are those of the epilogue's own sweep, also where it is subnormal."""
    from torch_dwconv import _C

    n, c, h, w, k, s, p = shape
    x, _, gy = (t.to(gpu) for t in make_inputs(shape, seed=17))
    x[:, 0] = x[:, 0].clamp(-1, 1) * 89
    wt = torch.zeros(c, 1, k, k, device=gpu)
    wt[:, :, p, p] = 1
    gx = _C.dwconv2d_fused_backward(x, gy, wt, None, None, "silu", s, s, p, p)[0]
    assert ",epi>" in _C.last_variant(), _C.last_variant()
    want = torch.zeros_like(x)
    want[:, :, ::s, ::s] = _C.dwconv2d_epilogue_backward(x[:, :, ::s, ::s].contiguous(), gy, None, None, "silu")[0]
    assert torch.equal(gx, want), float((gx - want).abs().max())


@pytest.mark.parametrize("act", [None, "relu", "relu6"])
@pytest.mark.parametrize("shape", [(2, 6, 14, 14, 3, 1, 1), (2, 3, 38, 38, 3, 2, 1), (2, 3, 56, 56, 5, 1, 2)], ids=shape_id)
def test_activations(gpu, shape, act):
    """Against the convolution, the epilogue's backward and the plain backward; without scale and shift too.  ReLU and ReLU6:
    inputs are small integers, so that every sum is exact and no output is on the other side of a corner."""
    from torch_dwconv import _C

    n, c, h, w, k, s, p = shape
    x, wt, gy = (t.mul(2).round().to(gpu) for t in make_inputs(shape, seed=5))
    for scale, shift in ((None, None), (torch.full((c,), 0.5, device=gpu), torch.full((c,), 1.25, device=gpu))):
        got = _C.dwconv2d_fused_backward(x, gy, wt, scale, shift, act, s, s, p, p)
        conv = _C.dwconv2d(x, wt, 1, 1, s, s, p, p, p, p, True)
        conv_grad, *sums = _C.dwconv2d_epilogue_backward(conv, gy, scale, shift, act)
        for a, b in zip(got, (*_C.dwconv2d_backward(x, conv_grad, wt, s, s, p, p), *sums)):
            torch.testing.assert_close(a, b, rtol=1e-5, atol=1e-5 * float(b.abs().max()))


@pytest.mark.parametrize("shape", [(1, 2, 13, 13, 3, 1, 1), (1, 2, 75, 75, 3, 1, 1), (1, 2, 75, 75, 5, 2, 2)], ids=shape_id)
def test_non_finite_inputs_stay_where_they_are(gpu, shape):
    """An infinity in the plane's last element reaches the in_grad elements that it reaches through the three separate calls,
    and no others: nothing beyond the plane is multiplied with it."""
    from torch_dwconv import _C

    n, c, h, w, k, s, p = shape
    x, wt, gy = (t.to(gpu) for t in make_inputs(shape, seed=9))
    scale, shift = params(c, gpu)
    x[:, :, -1, -1] = float("inf")
    gx, gw, s_scale, s_shift = _C.dwconv2d_fused_backward(x, gy, wt, scale, shift, "silu", s, s, p, p)
    conv_grad, *sums = _C.dwconv2d_epilogue_backward(_C.dwconv2d(x, wt, 1, 1, s, s, p, p, p, p, True), gy, scale, shift, "silu")
    want, gw_want = _C.dwconv2d_backward(x, conv_grad, wt, s, s, p, p)
    assert torch.equal(torch.isfinite(gx), torch.isfinite(want)) and not bool(torch.isfinite(want).all())
    assert not bool((torch.isfinite(gw_want) & ~torch.isfinite(gw)).any())
    assert torch.equal(torch.isfinite(s_scale), torch.isfinite(sums[0]))
    assert torch.equal(torch.isfinite(s_shift), torch.isfinite(sums[1]))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("shape", [(1, 2, 40, 36, 3, 1, 1), (1, 2, 56, 56, 3, 1, 1), (1, 2, 75, 75, 3, 1, 1), (1, 2, 75, 75, 5, 1, 2), (1, 2, 64, 129, 5, 1, 2),
                                   (1, 2, 112, 112, 3, 2, 1), (1, 2, 64, 64, 3, 2, 1), (1, 2, 75, 75, 5, 2, 2), (1, 2, 57, 64, 5, 2, 2)], ids=shape_id)
def test_infinite_input_reaches_its_own_taps_only(gpu, shape, dtype):
    """The tiled kernels: blocks that would hang over the plane's last row, or repeat a neighbour's rows, add nothing to the filter's
    gradient.  One infinite element of x, at either end of the plane or inside: the taps whose sums hold it are not finite, the others
    are, but for what the plain kernels have too: columns past a row that is not whole blocks of four (of two at stride 2)."""
    from torch_dwconv import _C

    n, c, h, w, k, s, p = shape
    x, wt, gy = (t.to(dtype).to(gpu) for t in make_inputs(shape, seed=19))
    for iy, ix in ((h - 1, w - 1), (0, 0), (h - 1, w // 2), (h // 2, w - 1), (h // 2, w // 2)):
        xi = x.clone()
        xi[:, :, iy, ix] = float("inf")
        gw = _C.dwconv2d_fused_backward(xi, gy, wt, None, None, None, s, s, p, p)[1]
        assert _C.last_variant().startswith("bwd_tile"), _C.last_variant()
        blocks = 4 // s
        got = (~torch.isfinite(gw)).cpu()
        rows, cols, wide = ([(i + p - t) % s == 0 and 0 <= (i + p - t) // s < e for t in range(k)]
                            for i, e in ((iy, gy.shape[2]), (ix, gy.shape[3]), (ix, -(-gy.shape[3] // blocks) * blocks)))
        own = torch.tensor([[r and q for q in cols] for r in rows]).expand(c, 1, k, k)
        most = torch.tensor([[r and q for q in wide] for r in rows]).expand(c, 1, k, k)
        assert bool((got | ~own).all()) and bool((most | ~got).all()), (iy, ix, gw)
        assert not bool((got & torch.isfinite(_C.dwconv2d_backward(xi, gy, wt, s, s, p, p)[1]).cpu()).any()), (iy, ix, gw)


@pytest.mark.parametrize("native", [True, False], ids=["native", "ctypes"])
def test_the_rest_takes_the_separate_calls(gpu, monkeypatch, native):
    from torch_dwconv import _C

    if not native:
        monkeypatch.setattr(_C, "_binding", _C._NoBinding())
    x, w = torch.randn(2, 4, 20, 20, device=gpu), torch.randn(4, 1, 7, 7, device=gpu)
    assert _C.dwconv2d_fused_backward(x, x, w, None, None, "silu", 1, 1, 3, 3) is None  # 7x7
    w = torch.randn(4, 1, 3, 3, device=gpu)
    assert _C.dwconv2d_fused_backward(x, torch.randn(2, 4, 18, 18, device=gpu), w, None, None, "silu", 1, 1, 0, 0) is None
    assert _C.dwconv2d_fused_backward(x.double(), x.double(), w.double(), None, None, "silu", 1, 1, 1, 1) is None
    y = x.contiguous(memory_format=torch.channels_last)
    assert _C.dwconv2d_fused_backward(y, y, w, None, None, "silu", 1, 1, 1, 1) is None
    for bad in (x[:1], x[:, :3], x.half(), x.cpu(), x[0]):
        assert _C.dwconv2d_fused_backward(x, bad, w, None, None, "silu", 1, 1, 1, 1) is None
    for bad in (torch.ones(3, device=gpu), torch.ones(4)):
        assert _C.dwconv2d_fused_backward(x, x, w, bad, None, "silu", 1, 1, 1, 1) is None
    assert _C.dwconv2d_fused_backward(x, x, w[:3], None, None, "silu", 1, 1, 1, 1) is None
    assert _C.dwconv2d_fused_backward(x, x, w, None, None, "gelu", 1, 1, 1, 1) is None
    assert _C.dwconv2d_fused_backward(x, x, w, None, None, "silu", 1, 1, 1, 1) is not None


def test_a_dispatch_mode_changes_nothing(gpu):
    """Under a mode the calls go through their Python forms: the same kernel, the same bits."""
    from torch.utils._python_dispatch import TorchDispatchMode

    from torch_dwconv import _C

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    n, c, h, w, k, s, p = shape = (2, 6, 28, 28, 5, 1, 2)
    x, wt, gy = (t.to(gpu) for t in make_inputs(shape, seed=37))
    scale, shift = params(c, gpu)
    plain = _C.dwconv2d_fused_backward(x, gy, wt, scale, shift, "silu", s, s, p, p)
    with Mode():
        moded = _C.dwconv2d_fused_backward(x, gy, wt, scale, shift, "silu", s, s, p, p)
    assert all(torch.equal(a, b) and a.stride() == b.stride() for a, b in zip(plain, moded))
