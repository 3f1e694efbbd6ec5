"""Two-element dot products keep subnormal numbers: 16-bit elements below the type's smallest normal one, and bfloat16 results below
fp32's, through every kernel family that uses them."""
import pytest
import torch

from shapes import make_inputs, shape_id

pytestmark = pytest.mark.gpu

# (shape, channels-last, forward variant, backward variant): what a variant has to hold
CASES = [((2, 5, 14, 14, 5, 1, 2), False, ",dot2>", ",dot2>"), ((2, 3, 19, 19, 3, 1, 1), False, ",dot2>", ",dot2>"),
         ((2, 3, 9, 75, 3, 1, 1), False, "tile_down16_dot2", "bwd_stack16<"), ((1, 3, 40, 96, 3, 1, 1), False, "tile_down16_dot2", "16"),
         ((2, 3, 19, 35, 5, 2, 2), False, "tile_down16_dot2", "16"), ((2, 2, 56, 56, 7, 1, 3), False, "16", "bwd_stack16<"),
         ((2, 64, 28, 28, 5, 1, 2), True, "nhwc_down16<k5,s1,fwd,7x4", "nhwc_bwd16<k5"), ((2, 64, 28, 28, 7, 1, 3), True, "nhwc_down16<k7,s1,fwd,7x4", "nhwc_bwd16<k7"),
         ((2, 64, 28, 28, 5, 2, 2), True, "nhwc_down16<k5", "nhwc_bwd16<k5,s2")]


@pytest.fixture(autouse=True)
def also_small_calls(monkeypatch):
    """(rows of any width: larger layers come to the 16-bit forward kernel by themselves)"""
    monkeypatch.setenv("DWCONV_TUNING", "1")
    monkeypatch.setenv("DWCONV_T16_ANY_MIN", "0")


def both_ways(gpu, x, wt, gy, shape, nhwc, variants):
    from torch_dwconv import _C, depthwise_conv2d

    s, p = shape[5:]
    fmt = torch.channels_last if nhwc else torch.contiguous_format
    xg, gyg, wg = x.to(gpu).contiguous(memory_format=fmt), gy.to(gpu).contiguous(memory_format=fmt), wt.to(gpu)
    y = depthwise_conv2d(xg, wg, stride=s, padding=p)
    assert variants[0] in _C.last_variant(), _C.last_variant()
    gx, gw = (_C.dwconv2d_backward_nhwc if nhwc else _C.dwconv2d_backward)(xg, gyg, wg, s, s, p, p)
    assert variants[1] in _C.last_variant(), _C.last_variant()
    return [t.cpu().double() for t in (y, gx, gw)]


def references(x, wt, gy, shape):
    s, p = shape[5:]
    x, wt, gy = x.double(), wt.double(), gy.double()
    return [torch.nn.functional.conv2d(x, wt, stride=s, padding=p, groups=shape[1]),
            torch.nn.grad.conv2d_input(x.shape, wt, gy, stride=s, padding=p, groups=shape[1]),
            torch.nn.grad.conv2d_weight(x, wt.shape, gy, stride=s, padding=p, groups=shape[1])]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: shape_id(c[0]) + ("_nhwc" if c[1] else ""))
def test_subnormal_elements(gpu, case, dtype):
    """x and the gradient hold subnormal elements only, whole multiples of the type's smallest number.  Taps are small whole powers of
    two and their quotients lift the results into the normal range; where they meet each other (the filter's gradient) x is lifted.
    |error| <= u |ref| + 2^-20 of the largest result: one rounding, and fp32 sums of some hundred products."""
    shape, nhwc, *variants = case
    n, c, h, w, k, s, p = shape
    least, count = (2.0 ** -133, 127) if dtype == torch.bfloat16 else (2.0 ** -24, 1023)
    lift = 2.0 ** 40 if dtype == torch.bfloat16 else 2.0 ** 4
    x, wt, gy = make_inputs(shape, seed=71)
    low = lambda t: ((t * count / 4).round().clamp(-count, count).double() * least).to(dtype)  # noqa: E731
    wt = ((wt * k * 8).round().clamp(-16, 16) * lift / 8).to(dtype)
    assert float(low(x).double().abs().max()) <= least * count
    u = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    got = both_ways(gpu, low(x), wt, low(gy), shape, nhwc, variants)[:2]
    want = references(low(x), wt, low(gy), shape)[:2]
    lifted = ((gy * 8).round().clamp(-31, 31) * lift / 8).to(dtype)
    got.append(both_ways(gpu, low(x), wt, lifted, shape, nhwc, variants)[2])
    want.append(references(low(x), wt, lifted, shape)[2])
    for a, b in zip(got, want):
        assert float(b.abs().max()) > 0
        assert bool(((a - b).abs() <= u * b.abs() + 2.0 ** -20 * b.abs().max() + least / 2).all()), float((a - b).abs().max() / b.abs().max())


@pytest.mark.parametrize("case", CASES, ids=lambda c: shape_id(c[0]) + ("_nhwc" if c[1] else ""))
def test_subnormal_results(gpu, case):
    """bfloat16 elements and taps in the normal range whose products and sums lie below fp32's smallest normal number: multiples of
    2^-149 in the sums (whole ones by the choice of the elements, so the sums are exact) and of 2^-133 in the results."""
    shape, nhwc, *variants = case
    x, wt, gy = make_inputs(shape, seed=72)
    x, gy = (((t * 8).round().clamp(-32, 32) * 2.0 ** -75).to(torch.bfloat16) for t in (x, gy))
    wt = ((wt * shape[4] * 4).round().clamp(-16, 16) * 2.0 ** -63).to(torch.bfloat16)
    got = both_ways(gpu, x, wt, gy, shape, nhwc, variants)[:2]
    for a, b in zip(got, references(x, wt, gy, shape)[:2]):
        assert 0 < float(b.abs().max()) < 2.0 ** -123
        assert bool(((a - b).abs() <= 2.0 ** -9 * b.abs() + 2.0 ** -134).all()), float((a - b).abs().max())
