"""Whole-plane kernels with 16-bit LDS images: every width class (even, odd and ragged rows, powers of two), runs that start off a
four-element boundary, filter tensors off a 32-bit one, and infinities at row and plane ends."""
import pytest
import torch

import oracle
from shapes import make_inputs, shape_id
from test_gpu_any_width_staging import UNIT, check, shifted

pytestmark = pytest.mark.gpu

# odd channel counts and planes: the runs of a call start on every element of a group of four
STRIDE1 = [(2, 3, 9, 2, 3, 1, 1), (3, 5, 5, 4, 5, 1, 2), (2, 7, 7, 6, 5, 1, 2), (2, 33, 7, 7, 5, 1, 2), (1, 5, 8, 8, 3, 1, 1), (2, 3, 9, 9, 7, 1, 3),
           (1, 9, 11, 11, 5, 1, 2), (2, 3, 13, 13, 3, 1, 1), (3, 20, 14, 14, 3, 1, 1), (2, 7, 15, 15, 5, 1, 2), (1, 3, 16, 16, 5, 1, 2),
           (2, 5, 19, 17, 3, 1, 1), (1, 7, 5, 19, 5, 1, 2), (2, 3, 19, 19, 7, 1, 3), (1, 3, 22, 22, 3, 1, 1), (2, 3, 12, 25, 5, 1, 2),
           (1, 5, 26, 26, 5, 1, 2), (2, 3, 28, 28, 7, 1, 3), (2, 5, 1, 28, 5, 1, 2), (1, 3, 31, 31, 3, 1, 1), (1, 3, 64, 32, 5, 1, 2)]
STRIDE2 = [(2, 3, 5, 4, 3, 2, 1), (2, 5, 7, 7, 5, 2, 2), (1, 7, 8, 8, 5, 2, 2), (3, 3, 9, 10, 7, 2, 3), (2, 9, 14, 14, 5, 2, 2), (2, 3, 13, 15, 3, 2, 1),
           (1, 5, 16, 16, 5, 2, 2), (2, 3, 19, 19, 5, 2, 2), (1, 3, 24, 24, 5, 2, 2), (2, 3, 27, 27, 3, 2, 1), (1, 5, 32, 32, 5, 2, 2), (1, 2, 30, 30, 7, 2, 3)]


def images16(dtype, k, s, w):
    """Which forward calls run on 16-bit images (dwconv_small_common.hpp)."""
    if s == 2:
        return True
    if dtype == torch.bfloat16:
        return (w % 2 == 0 or w >= 17) and not (k == 3 and w in (10, 12))
    return not (k == 3 and w % 2 and w < 10)


@pytest.mark.parametrize("by", [0, 1])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("shape", STRIDE1 + STRIDE2, ids=shape_id)
def test_against_64_bits(gpu, shape, dtype, by):
    from torch_dwconv import _C, depthwise_conv2d

    n, c, h, w, k, s, p = shape
    x, wt, gy = (t.to(dtype) for t in make_inputs(shape, seed=51))
    taps = shifted(wt, gpu, by)
    y_ref, gx_ref, gw_ref = oracle.torch_reference(x, wt, gy, s, p)
    y = depthwise_conv2d(x.to(gpu), taps, stride=s, padding=p)
    assert (",dot2>" in _C.last_variant()) == images16(dtype, k, s, w), _C.last_variant()
    check(y, y_ref, UNIT[dtype])
    if s == 1:
        gx, gw = _C.dwconv2d_backward(x.to(gpu), gy.to(gpu), taps, s, s, p, p)
        assert (",dot2>" in _C.last_variant()) != ((k, w) in ((3, 7), (7, 15))), _C.last_variant()
        check(gx, gx_ref, UNIT[dtype])
        check(gw, gw_ref, UNIT[dtype])
        gx2, gw2 = _C.dwconv2d_backward(x.to(gpu), gy.to(gpu), taps, s, s, p, p)
        assert torch.equal(gx, gx2) and torch.equal(gw, gw2)
        gx3 = _C.dwconv2d(gy.to(gpu), taps, 1, 1, 1, 1, p, p, p, p, False)  # grad-input on its own
        check(gx3, gx_ref, UNIT[dtype])


@pytest.mark.parametrize("shape", [(2, 4, 14, 14, 5, 1, 2), (2, 3, 28, 28, 3, 1, 1), (1, 3, 16, 16, 7, 1, 3), (2, 3, 14, 14, 5, 2, 2), (1, 3, 18, 18, 3, 2, 1)], ids=shape_id)
def test_infinite_elements_reach_their_windows_only(gpu, shape):
    from torch_dwconv import _C, depthwise_conv2d

    n, c, h, w, k, s, p = shape
    x, wt, gy = (t.to(torch.bfloat16) for t in make_inputs(shape, seed=52))
    wt = wt.abs() + 0.25  # (an infinite element gives an infinite result under every tap)
    inf = float("inf")
    x2 = x.clone()
    x2[0, 0, 3, 0] = x2[0, 1, 4, w - 1] = x2[n - 1, c - 1, h - 1, w // 2] = x2[n - 1, 0, 0, w // 2 + 1] = inf
    y = depthwise_conv2d(x2.to(gpu), wt.to(gpu), stride=s, padding=p).cpu()
    ref = torch.nn.functional.conv2d(x2.double(), wt.double(), stride=s, padding=p, groups=c)
    assert not bool(y.isnan().any()) and torch.equal(y.isinf(), ref.isinf())
    if s == 1:
        gy2 = gy.clone()
        gy2[0, 0, 3, 0] = gy2[0, 1, 4, w - 1] = gy2[n - 1, c - 1, h - 1, w // 2] = inf
        gx, gw = (t.cpu() for t in _C.dwconv2d_backward(x.to(gpu), gy2.to(gpu), wt.to(gpu), 1, 1, p, p))
        want = torch.nn.grad.conv2d_input(x.shape, wt.double(), gy2.double(), padding=p, groups=c)
        assert not bool(gx.isnan().any()) and torch.equal(gx.isinf(), want.isinf())
        # grad-weight: an infinite gradient at a row's end meets no input under the taps that reach past it
        gy3 = gy.clone()
        gy3[0, 0, 3, 0] = gy3[0, 1, 4, w - 1] = inf
        _, gw = _C.dwconv2d_backward(x.to(gpu), gy3.to(gpu), wt.to(gpu), 1, 1, p, p)
        for j in range(k):
            assert bool(gw[0, 0, :, j].isfinite().all()) == (j < p), j  # column 0 under tap j reads column j - p of x
            assert bool(gw[1, 0, :, j].isfinite().all()) == (j > p), j


@pytest.mark.parametrize("shape", [(2, 5, 14, 14, 5, 1, 2), (2, 5, 19, 19, 3, 1, 1), (1, 4, 32, 32, 5, 2, 2)], ids=shape_id)
def test_fused_epilogue(gpu, shape):
    from torch_dwconv import depthwise_conv2d_fused, _C

    n, c, h, w, k, s, p = shape
    x, wt, gy = (t.to(torch.float16) for t in make_inputs(shape, seed=53))
    scale, bias = torch.linspace(0.5, 1.5, c), torch.linspace(-0.3, 0.4, c)
    y = depthwise_conv2d_fused(x.to(gpu), wt.to(gpu), bias.to(gpu), scale.to(gpu), "silu", s, p)
    assert ",dot2>" in _C.last_variant(), _C.last_variant()
    conv = torch.nn.functional.conv2d(x.double(), wt.double(), stride=s, padding=p, groups=c)
    z = conv * scale.double().view(1, -1, 1, 1) + bias.double().view(1, -1, 1, 1)
    check(y, z * torch.sigmoid(z), UNIT[torch.float16])


# odd planes and odd channel counts: the runs of consecutive images start on different elements of a group of four
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("shape", [(6, 3, 19, 19, 5, 1, 2), (5, 5, 13, 13, 3, 1, 1), (7, 7, 9, 9, 7, 1, 3), (5, 9, 11, 17, 5, 1, 2), (5, 3, 15, 15, 5, 1, 2),
                                   (6, 5, 28, 28, 3, 1, 1), (5, 3, 31, 31, 7, 1, 3), (9, 40, 7, 7, 5, 1, 2)], ids=shape_id)
def test_several_images_a_wavefront(gpu, monkeypatch, shape, dtype):
    """One wavefront a channel group: the next image is fetched while one is worked on, sums go on from image to image."""
    from torch_dwconv import _C

    n, c, h, w, k, s, p = shape
    monkeypatch.setenv("DWCONV_TUNING", "1")
    monkeypatch.setenv("DWCONV_SMALL_WGRAD_WAVES", "1")
    x, wt, gy = (t.to(dtype) for t in make_inputs(shape, seed=54))
    gx, gw = _C.dwconv2d_backward(x.to(gpu), gy.to(gpu), wt.to(gpu), s, s, p, p)
    assert ",dot2>" in _C.last_variant() and _C.last_variant().endswith(" chunks1"), _C.last_variant()
    _, gx_ref, gw_ref = oracle.torch_reference(x, wt, gy, s, p)
    check(gx, gx_ref, UNIT[dtype])
    check(gw, gw_ref, UNIT[dtype])
