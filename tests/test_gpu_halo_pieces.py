"""Window tiles of one position subtile a wave at every window piece count (4, 5, 6 and 8 rounds of
16-byte loads a thread, 4 and 8 waves): int8 gives the implicit GEMM's bits, fp16 stays within fp32
accumulation of a float64 conv."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from aexrt_amd import kernels as K
from aexrt_amd import packing

pytestmark = pytest.mark.gpu


# a 4 x 16 (8 x 16 with 8 waves) tile's 6 x 18 (10 x 18) window has 108 (180) pixels of c / 8 pieces
@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("c,jn", [(16, 1), (32, 4), (48, 2), (64, 1), (80, 2), (96, 1), (112, 2), (128, 1)])
def test_int8(cuda, c, jn, waves):
    import torch

    n, h, w, oc = 2, 13, 37, 72
    g = torch.Generator(device="cuda").manual_seed(c)
    x = torch.randn((n, h, w, c), generator=g, device=cuda).half()
    rng = np.random.default_rng(c)
    wt = (rng.standard_normal((oc, c, 3, 3)) / np.sqrt(9 * c)).astype(np.float32)
    pc = K.prepare_conv(O.conv_desc(n, c, h, w, oc, 3, 1, 1), 52, K.SRC_LAYOUT_INT8,
                        packing.pack_conv_int8(wt, fp16_engine=True),
                        rng.uniform(-0.1, 0.1, oc).astype(np.float32), device=cuda)
    slots = K.new_slots(c, cuda)
    K.amax_slots(x, slots)
    outs = []
    try:
        for mode in (K.HALO_FORCE if waves == 4 else K.HALO_FORCE8, K.HALO_OFF):
            K.set_conv3x3_halo(mode, jn, 1, waves, 16, c) if mode != K.HALO_OFF else K.set_conv3x3_halo(mode)
            y = torch.full((n, h, w, oc), 5.0, dtype=torch.float16, device=cuda)
            K.conv2d(pc, x, y, x_slots=slots)
            torch.cuda.synchronize()
            outs.append(y.view(torch.int16))
    finally:
        K.set_conv3x3_halo()
    assert torch.equal(*outs)


# stride 2: 9 x 33 (17 x 33) window pixels
@pytest.mark.parametrize("c,jn,waves", [(c, jn, waves) for c, jn in ((8, 1), (16, 2), (24, 4), (32, 1), (40, 2))
                                        for waves in (4, 8)] + [(48, 1, 8)])
def test_fp16_stride2(cuda, c, jn, waves):
    import torch
    import torch.nn.functional as F

    n, h, w, oc = 2, 27, 61, 40
    g = torch.Generator(device="cuda").manual_seed(c)
    x = torch.randn((n, h, w, c), generator=g, device=cuda).half()
    rng = np.random.default_rng(c)
    wt = (rng.standard_normal((oc, c, 3, 3)) / np.sqrt(9 * c)).astype(np.float32)
    b = rng.uniform(-0.1, 0.1, oc).astype(np.float32)
    pc = K.prepare_conv(O.conv_desc(n, c, h, w, oc, 3, 2, 1), 5, K.SRC_RAW_F32, wt, b, device=cuda)
    y = torch.full((n, 14, 31, oc), 5.0, dtype=torch.float32, device=cuda)
    try:
        K.set_conv3x3_halo(K.HALO_FORCE if waves == 4 else K.HALO_FORCE8, jn, 1, waves, 16, c)
        K.conv2d(pc, x, y, flags=K.OUT_F32)
        torch.cuda.synchronize()
    finally:
        K.set_conv3x3_halo()
    xd = x.cpu().double().permute(0, 3, 1, 2)
    wd, bd = torch.from_numpy(wt.astype(np.float16)).double(), torch.from_numpy(b).double()
    ref = F.conv2d(xd, wd, bd, stride=2, padding=1)
    # any order of the 9 c products and the bias in fp32
    bound = (9 * c + 1) * 2.0 ** -24 * F.conv2d(xd.abs(), wd.abs(), bd.abs(), stride=2, padding=1)
    assert bool(((y.cpu().double().permute(0, 3, 1, 2) - ref).abs() <= bound).all())
