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
    assert (" anystart" in variant) == bool(w % 2 or by), variant
    _, gx_ref, gw_ref = oracle.torch_reference(x, wt, gy, s, p)
    check(gx, gx_ref, UNIT[dtype])
    check(gw, gw_ref, UNIT[dtype])
    gx2, gw2 = _C.dwconv2d_backward(shifted(x, gpu, by), shifted(gy, gpu, by), wt.to(gpu), s, s, p, p)
    assert torch.equal(gx, gx2) and torch.equal(gw, gw2)


# the last and first sizes of the rule that sends grad-input of rows on any element through LDS as one run an image
@pytest.mark.parametrize("shape,run", [((71, 42, 75, 75, 3, 1, 1), False), ((19, 157, 75, 75, 3, 1, 1), True), ((19, 100, 95, 95, 3, 1, 1), True),
                                       ((19, 100, 97, 97, 3, 1, 1), False), ((64, 173, 39, 39, 5, 1, 2), True), ((64, 173, 41, 41, 5, 1, 2), False),
                                       ((64, 242, 33, 33, 7, 1, 3), False), ((64, 161, 40, 41, 3, 1, 1), True), ((64, 75, 59, 60, 3, 1, 1), False)],
                         ids=lambda v: shape_id(v) if isinstance(v, tuple) else str(v))
def test_results_as_one_run_where_it_is_faster(gpu, monkeypatch, shape, run):
    """Both ways leave the same bits (those of a few planes are checked against 64 bits)."""
    from torch_dwconv import _C

    n, c, h, w, k, s, p = shape
    g = torch.Generator(gpu).manual_seed(63)
    x, gy = (torch.randn(n, c, h, w, device=gpu, generator=g).to(torch.bfloat16) for _ in range(2))
    wt = (torch.randn(c, 1, k, k, device=gpu, generator=g) / k).to(torch.bfloat16)
    gx, gw = _C.dwconv2d_backward(x, gy, wt, s, s, p, p)
    variant = _C.last_variant()
    assert variant.startswith("bwd_stack16<") and (" runout" in variant) == run, variant
    monkeypatch.setenv("DWCONV_TUNING", "1")
    monkeypatch.setenv("DWCONV_STACK_RUN", "0" if run else "1")
    gx2, gw2 = _C.dwconv2d_backward(x, gy, wt, s, s, p, p)
    assert (" runout" in _C.last_variant()) == (not run and k <= 5 and w % 2 != 0), _C.last_variant()
    assert torch.equal(gx, gx2) and torch.equal(gw, gw2)
    last = slice(c - 2, c)
    want = torch.nn.grad.conv2d_input((n, 2, h, w), wt[last].double().cpu(), gy[:, last].double().cpu(), padding=p, groups=2)
    check(gx[:, last], want, UNIT[torch.bfloat16])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("shape,by", [((5, 2, 34, 49, 3, 1, 1), 0), ((5, 2, 34, 50, 3, 1, 1), 1), ((2, 3, 9, 133, 3, 1, 1), 0), ((7, 1, 33, 33, 5, 1, 2), 0),
                                      ((33, 2, 36, 38, 5, 1, 2), 1), ((33, 3, 35, 51, 5, 1, 2), 0), ((3, 2, 130, 66, 3, 1, 1), 1)],
                         ids=lambda v: shape_id(v) if isinstance(v, tuple) else str(v))
def test_results_as_one_run(gpu, monkeypatch, shape, by, dtype):
    """Small tensors through the switch: remainders, shifted tensors, tiles that span images, one and many tiles a workgroup."""
    from torch_dwconv import _C

    n, c, h, w, k, s, p = shape
    x, wt, gy = (t.to(dtype) for t in make_inputs(shape, seed=64))
    args = (shifted(x, gpu, by), shifted(gy, gpu, by), wt.to(gpu), s, s, p, p)
    gx, gw = _C.dwconv2d_backward(*args)
    assert " runout" not in _C.last_variant(), _C.last_variant()
    monkeypatch.setenv("DWCONV_TUNING", "1")
    monkeypatch.setenv("DWCONV_STACK_RUN", "1")
    gx2, gw2 = _C.dwconv2d_backward(*args)
    assert " runout" in _C.last_variant(), _C.last_variant()
    assert torch.equal(gx, gx2) and torch.equal(gw, gw2)
    monkeypatch.setenv("DWCONV_STACK_WGS", "1")
    gx3, gw3 = _C.dwconv2d_backward(*args)
    assert " chunks1 " in _C.last_variant(), _C.last_variant()
    _, gx_ref, gw_ref = oracle.torch_reference(x, wt, gy, s, p)
    check(gx3, gx_ref, UNIT[dtype])
    check(gw3, gw_ref, UNIT[dtype])
    assert torch.equal(gx, gx3)


@pytest.mark.parametrize("shape,chunks", [((16, 64, 91, 91, 3, 1, 1), 24), ((8, 32, 193, 193, 3, 1, 1), 48), ((20, 64, 80, 80, 3, 1, 1), 24),
                                          ((64, 96, 33, 33, 3, 1, 1), 21), ((16, 64, 83, 83, 3, 1, 1), 28), ((64, 96, 45, 45, 3, 1, 1), 22)],
                         ids=lambda v: shape_id(v) if isinstance(v, tuple) else str(v))
def test_workgroups_that_share_the_tiles(gpu, shape, chunks):
    """3x3: up to 2048 workgroups where one of them then has fewer tiles than with 1536, and no more than those where it has not."""
    from torch_dwconv import _C

    n, c, h, w, k, s, p = shape
    x, wt, gy = (t.to(torch.bfloat16) for t in make_inputs(shape, seed=65))
    gx, gw = _C.dwconv2d_backward(x.to(gpu), gy.to(gpu), wt.to(gpu), s, s, p, p)
    assert f" chunks{chunks} " in _C.last_variant(), _C.last_variant()
    few = slice(0, 3)
    _, gx_ref, gw_ref = oracle.torch_reference(x[:, few], wt[few], gy[:, few], s, p)
    check(gx[:, few], gx_ref, UNIT[torch.bfloat16])
    check(gw[few], gw_ref, UNIT[torch.bfloat16])


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
