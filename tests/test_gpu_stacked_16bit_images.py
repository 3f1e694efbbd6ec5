"""Stacked backward kernel with 16-bit LDS images: infinities beside the windows, every remainder of a row by its four-column
blocks, rows on and off 32-bit boundaries, and tiles that span images and end inside one."""
import pytest
import torch

import oracle
from shapes import make_inputs, shape_id
from test_gpu_any_width_staging import UNIT, check, shifted

pytestmark = pytest.mark.gpu

SHAPES = [(5, 2, 34, w, k, 1, k // 2) for w in (48, 49, 50, 51) for k in (3, 5, 7) if (w, k) != (48, 7)] + [
    (2, 3, 9, 133, 3, 1, 1), (1, 2, 56, 56, 7, 1, 3), (7, 1, 33, 33, 5, 1, 2), (3, 2, 130, 66, 3, 1, 1), (33, 2, 36, 38, 5, 1, 2), (9, 3, 41, 43, 7, 1, 3), (64, 1, 11, 100, 7, 1, 3)]


@pytest.mark.parametrize("by", [0, 1])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("shape", SHAPES, ids=shape_id)
def test_backward(gpu, shape, dtype, by):
    from torch_dwconv import _C

    n, c, h, w, k, s, p = shape
    x, wt, gy = (t.to(dtype) for t in make_inputs(shape, seed=61))
    gx, gw = _C.dwconv2d_backward(shifted(x, gpu, by), shifted(gy, gpu, by), wt.to(gpu), s, s, p, p)
    variant = _C.last_variant()
    assert variant.startswith("bwd_stack16<") and " dot2" in variant, variant
    # rows that start on any element: grad-input leaves through LDS as one run an image
    assert (" anystart" in variant) == bool(w % 2 or by), variant
    _, gx_ref, gw_ref = oracle.torch_reference(x, wt, gy, s, p)
    check(gx, gx_ref, UNIT[dtype])
    check(gw, gw_ref, UNIT[dtype])
    gx2, gw2 = _C.dwconv2d_backward(shifted(x, gpu, by), shifted(gy, gpu, by), wt.to(gpu), s, s, p, p)
    assert torch.equal(gx, gx2) and torch.equal(gw, gw2)


@pytest.mark.parametrize("shape", [(2, 2, 48, 48, 3, 1, 1), (2, 2, 40, 51, 5, 1, 2), (2, 2, 40, 54, 7, 1, 3)], ids=shape_id)
def test_infinite_gradients_reach_their_windows_only(gpu, shape):
    from torch_dwconv import _C

    n, c, h, w, k, s, p = shape
    x, wt, gy = (t.to(torch.bfloat16) for t in make_inputs(shape, seed=62))
    wt = wt.abs() + 0.25
    gy[0, 0, 5, 0] = gy[0, 1, 9, w - 1] = gy[1, 1, h - 1, 17] = gy[1, 0, 0, 22] = float("inf")
    gx, _ = _C.dwconv2d_backward(x.to(gpu), gy.to(gpu), wt.to(gpu), 1, 1, p, p)
    assert _C.last_variant().startswith("bwd_stack16<"), _C.last_variant()
    want = torch.nn.grad.conv2d_input(x.shape, wt.double(), gy.double(), padding=p, groups=c)
    gx = gx.cpu()
    assert not bool(gx.isnan().any()) and torch.equal(gx.isinf(), want.isinf())
