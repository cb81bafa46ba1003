"""NHWC -> dense fp32 NCHW at the edges of its tiles (64 positions, up to 64 channels, 16-byte loads or
single elements), fp16 and fp32, on dense tensors and on slices that are not 16-byte aligned."""
from __future__ import annotations

import ctypes

import pytest

from aexrt_amd import _lib
from aexrt_amd import kernels as K

pytestmark = pytest.mark.gpu

CASES = [
    # n, h, w, c, channels of the tensor, first channel
    (1, 1, 1, 1, 1, 0),
    (2, 5, 7, 3, 3, 0),
    (1, 9, 7, 64, 64, 0),       # 63 positions
    (3, 13, 5, 65, 65, 0),      # 65 positions, 65 channels
    (2, 42, 50, 144, 144, 0),   # three tiles of 48 channels
    (2, 8, 8, 72, 96, 8),
    (2, 11, 13, 40, 63, 5),     # unaligned slice
    (1, 25, 21, 513, 520, 3),
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("half", [False, True])
def test_nhwc_to_nchw(cuda, case, half):
    import torch

    n, h, w, c, ct, c0 = case
    g = torch.Generator(device="cuda").manual_seed(c)
    whole = torch.randn((n, h, w, ct), generator=g, device=cuda).to(torch.float16 if half else torch.float32)
    y = torch.full((n, c, h, w), 9.0, device=cuda)
    x = whole[..., c0:c0 + c]
    v = _lib.TensorView(data=x.data_ptr(), n_stride=h * w * ct, c_stride=ct, amax_stripes=0, amax_slots=None,
                        amax_stripe_stride=0)
    _lib.check(_lib.lib().aexrt_hip_nhwc_to_nchw_f32(ctypes.byref(v), int(half), n, c, h * w, y.data_ptr(),
                                                      K._stream()), "nhwc_to_nchw_f32")
    assert torch.equal(y, x.permute(0, 3, 1, 2).float())
