"""Parity of kernels and dispatch rules at the sizes where they change hands:
tile edges, remainders, unaligned views, the smallest and largest of a range."""
from __future__ import annotations

import numpy as np
import pytest

from gpu_util import ctx, rounder, tdtype, vrs

pytestmark = pytest.mark.gpu
DT = [pytest.param(vrs.F32, id="f32"), pytest.param(vrs.BF16, id="bf16")]


@pytest.mark.parametrize("dtype", DT)
@pytest.mark.parametrize("n,c,c_pad,h,w,shift", [
    (2, 3, 8, 16, 32, 0),      # the 8-channel tile, one whole tile
    (1, 3, 8, 19, 27, 0),      # its last partial tile, single-pixel accesses (513 pixels)
    (1, 3, 3, 5, 7, 0),        # rows that no 16-byte chunk fits
    (2, 64, 64, 8, 8, 0),      # the 64-channel tile, one whole tile
    (1, 65, 72, 5, 13, 0),     # 65 pixels and channels: both remainders, padded rows
    (1, 130, 130, 4, 4, 1),    # unaligned rows and an image base off 16 bytes
])
def test_layout_conversions_exact(dtype, n, c, c_pad, h, w, shift):
    """NCHW float32 -> NHWC and back are copies (one rounding to the element type)."""
    import torch
    rng = np.random.default_rng(21)
    x = rng.standard_normal((n, c, h, w)).astype(np.float32)
    x[0, 0, 0, 0], x[0, -1, -1, -1] = np.inf, -0.0
    flat = torch.zeros(shift + x.size, device="cuda")
    xt = flat[shift:].view(n, c, h, w)
    xt.copy_(torch.from_numpy(x))
    y = torch.full((n, h, w, c_pad), 7.0, dtype=tdtype(dtype), device="cuda")
    ctx().pack_input(xt, vrs.nhwc(y), dtype)
    torch.cuda.synchronize()
    want = np.zeros((n, h, w, c_pad), np.float32)
    want[..., :c] = rounder(dtype)(x).transpose(0, 2, 3, 1)
    assert np.array_equal(y.float().cpu().numpy(), want)
    # back from a channel slice (offset 1 when there is room: unaligned) and from the whole buffer
    for off in (0, 1):
        back = torch.full((shift + n * (c - off) * h * w,), 9.0, device="cuda")
        ctx().unpack_output(vrs.nhwc(y, c - off, off), dtype, back[shift:].view(n, c - off, h, w))
        torch.cuda.synchronize()
        assert np.array_equal(back[shift:].cpu().numpy().reshape(n, c - off, h, w), rounder(dtype)(x)[:, off:])
