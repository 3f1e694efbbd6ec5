"""The 16-bit tiled forward kernel on rows of any width: every remainder of a row by its blocks, rows and tensors that start on
and off 32-bit boundaries, one and several planes to a workgroup, bands that end inside a block, and infinities at row ends."""
import pytest
import torch

import oracle
from shapes import make_inputs, shape_id
from test_gpu_any_width_staging import UNIT, check, shifted

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def also_small_calls(request, monkeypatch):
    """These layers are smaller than those that come to this kernel by themselves (see test_which_calls)."""
    if "own_rule" not in request.keywords:
        monkeypatch.setenv("DWCONV_TUNING", "1")
        monkeypatch.setenv("DWCONV_T16_ANY_MIN", "0")


# stride 2: blocks of four results; stride 1: blocks of eight
SHAPES = [(2, 3, 9, 30 + w, 3, 2, 1) for w in range(3, 10)] + [(1, 3, 6, 64 + w, 3, 1, 1) for w in (1, 3, 5, 7)] + [
    (1, 2, 5, 128 + w, 5, 1, 2) for w in (1, 2, 6)] + [(2, 2, 10, 56 + w, 7, 1, 3) for w in (1, 2, 3, 5, 6, 7)] + [
    (3, 5, 33, 33, 3, 2, 1), (2, 7, 35, 37, 5, 2, 2), (1, 3, 1, 75, 3, 1, 1), (1, 2, 2, 49, 7, 2, 3), (1, 2, 150, 150, 3, 2, 1),
    (2, 1, 75, 75, 5, 2, 2), (1, 3, 131, 131, 5, 1, 2), (1, 1, 3, 901, 3, 2, 1), (2, 3, 150, 150, 3, 1, 1), (1, 2, 64, 36, 3, 2, 1)]


@pytest.mark.parametrize("by", [0, 1, 3])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("shape", SHAPES, ids=shape_id)
def test_forward(gpu, shape, dtype, by):
    from torch_dwconv import depthwise_conv2d, _C

    n, c, h, w, k, s, p = shape
    x, wt, gy = (t.to(dtype) for t in make_inputs(shape, seed=31))
    y = depthwise_conv2d(shifted(x, gpu, by), wt.to(gpu), stride=s, padding=p)
    variant = _C.last_variant()
    assert variant.startswith("tile_down16_dot2") and variant.endswith(" runout anywidth"), variant
    check(y, oracle.torch_reference(x, wt, gy, s, p)[0], UNIT[dtype])


@pytest.mark.parametrize("shape", [(2, 3, 9, 75, 3, 1, 1), (2, 3, 19, 35, 3, 2, 1), (2, 2, 11, 37, 5, 2, 2), (1, 2, 9, 59, 7, 1, 3)], ids=shape_id)
def test_infinite_inputs_reach_their_windows_only(gpu, shape):
    """What a row's last load reads of the next row, and the partner of an unpaired tap, take no part in any result."""
    from torch_dwconv import depthwise_conv2d

    n, c, h, w, k, s, p = shape
    x, wt, gy = (t.to(torch.bfloat16) for t in make_inputs(shape, seed=32))
    wt = wt.abs() + 0.25  # (an infinite element gives an infinite result under every tap)
    x[0, 0, 3, 0] = x[0, 1, 4, w - 1] = x[n - 1, 0, 5, w // 2] = float("inf")
    y = depthwise_conv2d(x.to(gpu), wt.to(gpu), stride=s, padding=p).cpu()
    ref = torch.nn.functional.conv2d(x.double(), wt.double(), stride=s, padding=p, groups=c)
    assert not bool(y.isnan().any())
    assert torch.equal(y.isinf(), ref.isinf())


@pytest.mark.parametrize("shape", [(2, 3, 13, 75, 3, 1, 1), (2, 3, 13, 35, 3, 2, 1), (1, 3, 9, 59, 7, 1, 3)], ids=shape_id)
def test_fused_epilogue_and_grad_input(gpu, shape):
    from torch_dwconv import depthwise_conv2d_fused, _C

    n, c, h, w, k, s, p = shape
    x, wt, gy = (t.to(torch.bfloat16) for t in make_inputs(shape, seed=33))
    scale, bias = torch.linspace(0.5, 1.5, c), torch.linspace(-0.3, 0.4, c)
    y = depthwise_conv2d_fused(x.to(gpu), wt.to(gpu), bias.to(gpu), scale.to(gpu), "silu", s, p)
    assert _C.last_variant().endswith(" runout anywidth"), _C.last_variant()
    conv = torch.nn.functional.conv2d(x.double(), wt.double(), stride=s, padding=p, groups=c)
    z = conv * scale.double().view(1, -1, 1, 1) + bias.double().view(1, -1, 1, 1)
    check(y, z * torch.sigmoid(z), UNIT[torch.bfloat16])
    if s == 1:
        gx = _C.dwconv2d(gy.to(gpu), wt.to(gpu), 1, 1, 1, 1, p, p, p, p, False)
        assert _C.last_variant().endswith(" runout anywidth"), _C.last_variant()
        check(gx, oracle.torch_reference(x, wt, gy, s, p)[1], UNIT[torch.bfloat16])


# the last and first sizes of the rule that keeps small calls on the kernels of before
@pytest.mark.own_rule
@pytest.mark.parametrize("shape,here", [((9, 31, 75, 75, 3, 1, 1), False), ((7, 40, 75, 75, 3, 1, 1), True), ((1, 233, 150, 150, 5, 1, 2), False),
                                        ((3, 78, 150, 150, 5, 1, 2), True), ((13, 37, 66, 66, 7, 1, 3), False), ((2, 241, 66, 66, 7, 1, 3), True),
                                        ((8, 31, 65, 65, 7, 1, 3), False), ((3, 83, 65, 65, 7, 1, 3), True), ((9, 31, 75, 75, 3, 2, 1), False),
                                        ((7, 40, 75, 75, 3, 2, 1), True), ((1, 3, 150, 150, 3, 2, 1), True), ((6, 31, 75, 75, 5, 2, 2), False),
                                        ((11, 17, 75, 75, 5, 2, 2), True), ((1, 2, 9, 131, 5, 2, 2), True), ((1, 359, 54, 54, 7, 2, 3), False),
                                        ((1, 360, 54, 54, 7, 2, 3), True), ((1, 2, 9, 37, 7, 2, 3), True)],
                         ids=lambda v: shape_id(v) if isinstance(v, tuple) else str(v))
def test_which_calls(gpu, shape, here):
    from torch_dwconv import depthwise_conv2d, _C

    n, c, h, w, k, s, p = shape
    x, wt, gy = (t.to(torch.bfloat16) for t in make_inputs(shape, seed=34))
    y = depthwise_conv2d(x.to(gpu), wt.to(gpu), stride=s, padding=p)
    variant = _C.last_variant()
    assert (variant.startswith("tile_down16_dot2") and variant.endswith(" runout anywidth")) == here, variant
    check(y, torch.nn.functional.conv2d(x.double(), wt.double(), stride=s, padding=p, groups=c), UNIT[torch.bfloat16])
