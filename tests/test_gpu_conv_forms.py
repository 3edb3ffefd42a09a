"""The closure convolution at the sizes where its form changes: one tile per
workgroup up to four 32-pixel tiles per CU, above that strips of rows per
wave (32 channels; with a shorter last segment, with wrapped halos of the
smallest height) or the LDS forms (8 channels).

Bars: FP32 accumulation of 800 BF16 products, each exact in FP32: with
terms of standard deviation 0.2 the sums are about 6 and the largest about
30, the rounding of 800 additions (relative 6e-8 of the partial sums, random
signs) below 1e-5 of the largest. The fused epilogues of a shape use the
same accumulation, so they agree with the unfused composition in every bit.
"""

import numpy as np
import pytest
import torch

from oracle import cnn as C
from fluidsim_amd import _lib
from fluidsim_amd.closure import bf16_bits, bf16_value

pytestmark = pytest.mark.gpu

SHAPES = [(1, 4, 32), (2, 4, 96), (8, 128, 32), (9, 116, 32), (300, 4, 32), (50, 92, 32)]


@pytest.mark.parametrize("ci", [8, 32])
@pytest.mark.parametrize("shape", SHAPES)
def test_convolution_forms(ci, shape):
    rng = np.random.default_rng(5)
    B, H, W = shape
    x = rng.standard_normal(shape + (ci,))
    w = rng.standard_normal((32, 25, ci)) * 0.2
    b = rng.standard_normal(32).astype(np.float32)
    # the oracle on the first, a middle and the last image
    pick = sorted({0, B // 2, B - 1})
    value = lambda a: bf16_value(bf16_bits(a)).astype(np.float64)
    # one float past a 16-byte boundary: bias and outputs need 4-byte alignment
    flat = torch.zeros(1 + 32 + B * H * W * 32, dtype=torch.float32, device="cuda")
    bd = flat[1:33]
    bd.copy_(torch.from_numpy(b))
    xd = torch.from_numpy(bf16_bits(x)).cuda()
    wd = torch.from_numpy(bf16_bits(w)).cuda()
    s = _lib.stream_ptr()
    args = (_lib.dptr(xd), B, H, W, ci, _lib.dptr(wd), _lib.dptr(bd))
    for co in (32, 8, 3, 1):
        y = flat[33:33 + B * H * W * co].view(B, H, W, co)
        _lib.call("fsx_cnn_conv_fwd", *args, co, _lib.dptr(y), s)
        ref = C.conv(value(x[pick]), value(w), b.astype(np.float64), co)
        got = y[pick].cpu().numpy()
        assert np.abs(got - ref).max() < 1e-5 * np.abs(ref).max()
        if co == 32:
            pre = y.clone()
    act = lambda: torch.zeros((B, H, W, 32), dtype=torch.int16, device="cuda")
    a0, a1, a2, d0, d1 = act(), act(), act(), act(), act()
    _lib.call("fsx_cnn_act", _lib.dptr(pre), B * H * W, 32, 32, 1, _lib.dptr(a0), s)
    y1 = torch.full_like(pre, np.nan)
    _lib.call("fsx_cnn_conv_fwd_act", *args, _lib.dptr(y1), _lib.dptr(a1), s)
    _lib.call("fsx_cnn_conv_fwd_act", *args, None, _lib.dptr(a2), s)
    assert torch.equal(pre, y1) and torch.equal(a0, a1) and torch.equal(a0, a2)
    other = torch.randn_like(pre)
    _lib.call("fsx_cnn_act_bwd", _lib.dptr(pre), 32, _lib.dptr(other), B * H * W, 32,
              _lib.dptr(d0), s)
    _lib.call("fsx_cnn_conv_bwd_act", *args, _lib.dptr(other), _lib.dptr(d1), s)
    assert torch.equal(d0, d1)


@pytest.mark.parametrize("ci, shape", [(32, (1, 4, 288)), (32, (8, 16, 288)), (32, (2, 4, 1216)),
                                       (8, (2, 4, 1888)), (8, (40, 4, 1152))])
def test_wide_images(ci, shape):
    """Widths beyond what the patch rows of an LDS form could hold (at one row
    per workgroup 276 columns of 32 channels, 1884 of 8) run in the forms
    without LDS patches, and a wide 8-channel image in the LDS form; same bar as
    above."""
    rng = np.random.default_rng(6)
    B, H, W = shape
    x = rng.standard_normal(shape + (ci,))
    w = rng.standard_normal((32, 25, ci)) * 0.2
    b = rng.standard_normal(32).astype(np.float32)
    value = lambda a: bf16_value(bf16_bits(a)).astype(np.float64)
    xd, wd = (torch.from_numpy(bf16_bits(a)).cuda() for a in (x, w))
    bd = torch.from_numpy(b).cuda()
    y = torch.full((B, H, W, 32), np.nan, dtype=torch.float32, device="cuda")
    a = torch.zeros((B, H, W, 32), dtype=torch.int16, device="cuda")
    args = (_lib.dptr(xd), B, H, W, ci, _lib.dptr(wd), _lib.dptr(bd))
    _lib.call("fsx_cnn_conv_fwd_act", *args, _lib.dptr(y), _lib.dptr(a), _lib.stream_ptr())
    pick = sorted({0, B - 1})
    ref = C.conv(value(x[pick]), value(w), b.astype(np.float64), 32)
    assert np.abs(y[pick].cpu().numpy() - ref).max() < 1e-5 * np.abs(ref).max()
    act = torch.zeros_like(a)
    _lib.call("fsx_cnn_act", _lib.dptr(y), B * H * W, 32, 32, 1, _lib.dptr(act),
              _lib.stream_ptr())
    assert torch.equal(act, a)


def test_too_wide_for_the_staged_patch():
    """8 channels beyond a few tiles: the LDS form's width limit."""
    x = torch.zeros((512, 4, 1216, 8), dtype=torch.int16, device="cuda")
    w = torch.zeros((32, 25, 8), dtype=torch.int16, device="cuda")
    b = torch.zeros(32, dtype=torch.float32, device="cuda")
    y = torch.zeros((512, 4, 1216, 32), dtype=torch.float32, device="cuda")
    with pytest.raises(ValueError, match="too wide"):
        _lib.call("fsx_cnn_conv_fwd", _lib.dptr(x), 512, 4, 1216, 8, _lib.dptr(w), _lib.dptr(b),
                  32, _lib.dptr(y), _lib.stream_ptr())
