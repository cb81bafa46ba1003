"""fp16 1x1 convs without a measured tile, around the lines of their tile rule (96, 256 and 384 tiles, four
64-channel steps for the k split): within fp32 accumulation of a float64 product, on dense tensors and channel
slices, and the forced tile where one is set."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from aexrt_amd import kernels as K

pytestmark = pytest.mark.gpu

CASES = [
    # n, c, h, w, oc, slice of the input
    (1, 8, 1, 1, 8, None),
    (1, 304, 3, 5, 40, None),        # k split
    (3, 248, 31, 33, 16, (256, 8)),  # 49 tiles of a subtile, fewer than four k steps
    (8, 64, 39, 39, 24, None),       # 96 position tiles of two subtiles
    (8, 120, 64, 64, 56, None),      # 256
    (12, 72, 64, 65, 136, None),     # 390 of eight channel subtiles' two tiles
    (16, 264, 51, 51, 48, (272, 0)),
]


@pytest.mark.parametrize("case", CASES)
def test_within_fp32_accumulation(cuda, case):
    import torch

    n, c, h, w, oc, xs = case
    ct, c0 = xs or (c, 0)
    g = torch.Generator(device="cuda").manual_seed(c + oc)
    x = torch.randn((n, h, w, ct), generator=g, device=cuda).half()[..., c0:c0 + c]
    rng = np.random.default_rng(oc)
    wt = (rng.standard_normal((oc, c, 1, 1)) / np.sqrt(c)).astype(np.float32)
    b = rng.uniform(-0.1, 0.1, oc).astype(np.float32)
    pc = K.prepare_conv(O.conv_desc(n, c, h, w, oc, 1, 1, 0), 5, K.SRC_RAW_F32, wt, b, device=cuda)
    xd = x.cpu().double().reshape(-1, c)
    wd = torch.from_numpy(wt.reshape(oc, c).astype(np.float16)).double()
    ref = xd @ wd.t() + torch.from_numpy(b).double()
    # any order of the c products and the bias in fp32
    bound = (c + 1) * 2.0 ** -24 * (xd.abs() @ wd.abs().t() + torch.from_numpy(b).double().abs())
    try:
        for tile in ((0, 0), (2, 4)):
            K.set_conv_tile(*tile)
            y = torch.full((n, h, w, oc), 9.0, dtype=torch.float32, device=cuda)
            K.conv2d(pc, x, y, flags=K.OUT_F32)
            torch.cuda.synchronize()
            assert bool(((y.cpu().double().reshape(-1, oc) - ref).abs() <= bound).all())
    finally:
        K.set_conv_tile()
