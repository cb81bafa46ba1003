"""The fp32 conv at the edges of its tiles (64 positions x 4, 2 or 1 output channels, 8-channel steps of
the 1x1) against the oracle, without SiLU bit for bit; weights that are not finite and biases of -0,
where a tap outside the input must be left out, not multiplied by zero."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest

import oracle as O
from aexrt_amd import _lib

pytestmark = pytest.mark.gpu


def _conv(cuda, x, w, b, desc):
    import torch

    xd, wd, bd = (torch.from_numpy(np.ascontiguousarray(v, np.float32)).to(cuda) for v in (x, w, b))
    y = torch.empty(tuple(O.out_shape(desc)), dtype=torch.float32, device=cuda)
    d = _lib.ConvDesc.from_params(desc)
    _lib.check(_lib.lib().aexrt_hip_conv2d_f32(ctypes.byref(d), 0, xd.data_ptr(), wd.data_ptr(), bd.data_ptr(),
                                               y.data_ptr(), None), "conv2d_f32")
    torch.cuda.synchronize()
    return y.cpu().numpy()


CASES = [
    # n, c, h, w, oc, k, s, p, dilation, groups
    (1, 1, 1, 1, 1, 3, 1, 1, 1, 1),
    (3, 5, 7, 9, 5, 3, 1, 1, 1, 1),       # 189 positions: not a multiple of 64, OC % 4 == 1
    (2, 6, 13, 5, 8, 3, 2, 1, 1, 2),      # groups of 3 -> 4 channels
    (2, 6, 8, 8, 6, 3, 1, 1, 1, 6),       # one output channel to a group
    (1, 4, 8, 8, 4, 3, 1, 2, 2, 2),       # two, dilation 2
    (1, 7, 9, 33, 3, 1, 1, 0, 1, 1),      # 1x1: fewer channels than a step
    (2, 17, 9, 8, 20, 1, 2, 0, 1, 1),     # two steps and one channel over, stride 2
    (1, 8, 6, 6, 4, 1, 1, 1, 1, 1),       # padded 1x1: border positions are the bias
    (1, 3, 11, 12, 7, 5, 1, 2, 1, 1),     # 5x5: the kernel for any size
    (1, 9, 8, 8, 130, 3, 1, 1, 1, 1),     # several blocks of channel tiles
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("odd", ["plain", "inf_weight", "nan_weight", "minus_zero"])
def test_fp32_conv_sizes_bit_exact(cuda, case, odd):
    n, c, h, w, oc, k, s, p, d, g = case
    rng = np.random.default_rng(c * 100 + oc)
    desc = O.conv_desc(n, c, h, w, oc, k, s, p, dilation=d, groups=g)
    x = rng.standard_normal((n, c, h, w)).astype(np.float32)
    wt = rng.standard_normal((oc, c // g, k, k)).astype(np.float32)
    b = rng.uniform(-1, 1, oc).astype(np.float32)
    if odd == "inf_weight":
        wt[0, 0, 0, 0] = np.inf
    elif odd == "nan_weight":
        wt[-1, -1, -1, -1] = np.nan
    elif odd == "minus_zero":
        b[:] = -0.0
        x[:, :, : h // 2 + 1] = -0.0
        wt = np.abs(wt)
    got, want = _conv(cuda, x, wt, b, desc), O.cpu_conv2d(x, wt, b, desc, silu=False)
    nan = np.isnan(want)
    np.testing.assert_array_equal(np.isnan(got), nan)
    np.testing.assert_array_equal(got.view(np.uint32)[~nan], want.view(np.uint32)[~nan])
