"""16-bit channels-last kernels that take two taps or two pixels at a time: the 5x5 and 7x7 sweeps for both gradients and the
tall forward blocks, where a block, a channel group or a pair ends, and with infinities beside the windows."""
import pytest
import torch

import oracle
from shapes import make_inputs, shape_id

pytestmark = pytest.mark.gpu

# 7x7: from 2^15 elements on; blocks of 4 x 4 (backward), 7 x 4 or 4 x 4 (forward).  5x5: blocks of 7 x 2 and 7 x 4; stride 2, from
# 2^15 elements on and on even extents: 4 x 2 pixels of out_grad
CASES = [((2, 96, 13, 15, 7, 1, 3), "nhwc_bwd16<k7"), ((1, 768, 7, 7, 7, 1, 3), "nhwc_bwd16<k7"), ((3, 36, 28, 12, 7, 1, 3), "nhwc_bwd16<k7"),
         ((5, 132, 9, 6, 7, 1, 3), "nhwc_bwd16<k7"), ((1, 8, 64, 65, 7, 1, 3), "nhwc_bwd16<k7"), ((40, 840, 1, 1, 7, 1, 3), "nhwc_bwd16<k7"),
         ((2, 64, 16, 15, 7, 1, 3), "nhwc_down16<k7"), ((2, 68, 14, 13, 5, 1, 2), "nhwc_bwd16<k5"), ((9, 32, 7, 8, 5, 1, 2), "nhwc_bwd16<k5"),
         ((2, 64, 18, 18, 5, 2, 2), "nhwc_bwd16<k5,s2"), ((1, 36, 34, 30, 5, 2, 2), "nhwc_bwd16<k5,s2"), ((3, 132, 2, 46, 5, 2, 2), "nhwc_bwd16<k5,s2"),
         ((5, 100, 36, 2, 5, 2, 2), "nhwc_bwd16<k5,s2"), ((2, 64, 17, 18, 5, 2, 2), "nhwc_up216<k5"), ((2, 68, 14, 26, 3, 2, 1), "nhwc_bwd16<k3,s2"),
         ((1, 100, 21, 3, 5, 1, 2), "nhwc_bwd16<k5"), ((1, 12, 35, 1, 5, 1, 2), "nhwc_bwd16<k5")]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: shape_id(c[0]))
def test_both_directions(gpu, case, dtype):
    """|error| <= u |ref| + 1e-5 of the largest result: one rounding to the element type and fp32 sums."""
    from torch_dwconv import _C, depthwise_conv2d

    shape, backward = case
    n, c, h, w, k, s, p = shape
    x, wt, gy = (t.to(dtype) for t in make_inputs(shape, seed=41))
    xg, gyg = (t.to(gpu).contiguous(memory_format=torch.channels_last) for t in (x, gy))
    y = depthwise_conv2d(xg, wt.to(gpu), stride=s, padding=p)
    gx, gw = _C.dwconv2d_backward_nhwc(xg, gyg, wt.to(gpu), s, s, p, p)
    assert _C.last_variant().startswith(backward), _C.last_variant()
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for got, ref in zip((y, gx, gw), oracle.torch_reference(x, wt, gy, s, p)):
        assert got.shape == ref.shape
        err = (got.cpu().double() - ref).abs()
        assert bool((err <= u * ref.abs() + 1e-5 * ref.abs().max()).all()), float(err.max())
    gx2, gw2 = _C.dwconv2d_backward_nhwc(xg, gyg, wt.to(gpu), s, s, p, p)
    assert torch.equal(gx, gx2) and torch.equal(gw, gw2)


@pytest.mark.parametrize("k", [5, 7])
def test_infinite_elements_reach_their_windows_only(gpu, k):
    from torch_dwconv import _C, depthwise_conv2d

    n, c, h, w, p = 2, 64, 28, 28, k // 2
    x, wt, gy = (t.to(torch.bfloat16) for t in make_inputs((n, c, h, w, k, 1, p), seed=42))
    wt = wt.abs() + 0.25  # (an infinite element gives an infinite result under every tap)
    gy2 = gy.clone()
    x[0, 3, 9, 11] = x[1, 0, 0, 0] = gy2[1, 5, 14, 13] = gy2[0, 63, 27, 27] = float("inf")
    xg, gyg = (t.to(gpu).contiguous(memory_format=torch.channels_last) for t in (x, gy2))
    y = depthwise_conv2d(xg, wt.to(gpu), stride=1, padding=p).cpu()
    gx, _ = _C.dwconv2d_backward_nhwc(xg, gyg, wt.to(gpu), 1, 1, p, p)
    ref = torch.nn.functional.conv2d(x.double(), wt.double(), padding=p, groups=c)
    gx_ref = torch.nn.grad.conv2d_input(x.shape, wt.double(), gy2.double(), padding=p, groups=c)
    for got, want in ((y, ref), (gx.cpu(), gx_ref)):
        assert not bool(got.isnan().any())
        assert torch.equal(got.isinf(), want.isinf())


@pytest.mark.parametrize("k", [3, 5])
def test_infinite_gradients_of_stride_2_layers(gpu, k):
    """The transposed taps go in pairs of their own classes: no result takes a pixel of out_grad under a tap it does not have."""
    from torch_dwconv import _C

    n, c, h, w, p = 2, 64, 28, 28, k // 2
    x, wt, gy = (t.to(torch.bfloat16) for t in make_inputs((n, c, h, w, k, 2, p), seed=43))
    wt = wt.abs() + 0.25
    gy[1, 5, 7, 6] = gy[0, 63, 13, 13] = gy[0, 0, 0, 0] = gy[1, 8, 4, 13] = float("inf")
    xg, gyg = (t.to(gpu).contiguous(memory_format=torch.channels_last) for t in (x, gy))
    gx, _ = _C.dwconv2d_backward_nhwc(xg, gyg, wt.to(gpu), 2, 2, p, p)
    assert _C.last_variant().startswith(f"nhwc_bwd16<k{k},s2"), _C.last_variant()
    want = torch.nn.grad.conv2d_input(x.shape, wt.double(), gy.double(), stride=2, padding=p, groups=c)
    gx = gx.cpu()
    assert not bool(gx.isnan().any()) and torch.equal(gx.isinf(), want.isinf())


# heights that are not whole blocks of four rows, and two that are: the block that hangs over the map has zeros for out_grad there
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("shape", [(3, 64, 14, 16, 7, 1, 3), (3, 64, 13, 16, 7, 1, 3), (3, 36, 23, 20, 7, 1, 3), (40, 64, 2, 8, 7, 1, 3), (80, 64, 1, 8, 7, 1, 3),
                                   (3, 64, 16, 16, 7, 1, 3), (3, 64, 14, 16, 5, 2, 2), (3, 36, 26, 20, 5, 2, 2), (40, 64, 2, 8, 5, 2, 2), (3, 64, 16, 16, 5, 2, 2)],
                         ids=shape_id)
def test_infinite_input_reaches_its_own_taps_only(gpu, shape, dtype):
    """One infinite element of x a channel, in every row of the map's lower end and some others: the taps of the filter's gradient
    whose sums hold it are not finite, all others are.  (The widths are whole blocks.)"""
    from torch_dwconv import _C

    n, c, h, w, k, s, p = shape
    x, wt, gy = (t.to(dtype) for t in make_inputs(shape, seed=44))
    oh, ow = gy.shape[2:]
    own = torch.zeros(c, 1, k, k, dtype=torch.bool)
    for i in range(c):
        iy, ix = max(0, h - 1 - i % 8), (5 * i) % w
        x[i % n, i, iy, ix] = float("inf")
        for t in range(k):
            for u in range(k):
                oy, ox = iy + p - t, ix + p - u
                own[i, 0, t, u] = oy % s == 0 and ox % s == 0 and 0 <= oy // s < oh and 0 <= ox // s < ow
    xg, gyg = (t.to(gpu).contiguous(memory_format=torch.channels_last) for t in (x, gy))
    gw = _C.dwconv2d_backward_nhwc(xg, gyg, wt.to(gpu), s, s, p, p)[1].cpu()
    assert _C.last_variant().startswith(f"nhwc_bwd16<k{k},s{s}"), _C.last_variant()
    assert torch.equal(~gw.isfinite(), own)


# channel counts off the lane groups, maps off the blocks, images that end between two trips
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("shape", [(5, 40, 23, 17, 7, 1, 3), (5, 64, 28, 28, 7, 1, 3), (5, 40, 23, 17, 5, 1, 2), (40, 132, 7, 7, 5, 1, 2),
                                   (5, 36, 34, 30, 5, 2, 2), (5, 40, 28, 28, 3, 2, 1), (7, 36, 32, 20, 3, 1, 1)], ids=shape_id)
def test_several_trips_a_workgroup(gpu, monkeypatch, shape, dtype):
    """One workgroup a channel group: it carries its sums through every block of every image, and its views to later images."""
    from torch_dwconv import _C

    n, c, h, w, k, s, p = shape
    monkeypatch.setenv("DWCONV_TUNING", "1")
    monkeypatch.setenv("DWCONV_NHWC_WGRAD_WGS", "1")
    x, wt, gy = (t.to(dtype) for t in make_inputs(shape, seed=45))
    xg, gyg = (t.to(gpu).contiguous(memory_format=torch.channels_last) for t in (x, gy))
    gx, gw = _C.dwconv2d_backward_nhwc(xg, gyg, wt.to(gpu), s, s, p, p)
    variant = _C.last_variant()
    assert variant.startswith(f"nhwc_bwd16<k{k},s{s}") and variant.endswith(" chunks1"), variant
    rows, columns = (int(v) for v in variant.split(">")[0].split(",")[-1].split("x"))  # a block of out_grad
    lanes_c = int(variant.split(" lanes_c")[1].split(" ")[0])
    oh, ow = gy.shape[2:]
    blocks = n * -(-oh // rows) * -(-ow // columns)
    assert blocks >= 3 * (256 // lanes_c), variant
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for got, ref in zip((gx, gw), oracle.torch_reference(x, wt, gy, s, p)[1:]):
        err = (got.cpu().double() - ref).abs()
        assert bool((err <= u * ref.abs() + 1e-5 * ref.abs().max()).all()), float(err.max())
