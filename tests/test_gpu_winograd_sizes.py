"""The Winograd conv at the edges of its tiles and for each of its block shapes (16 tiles x 64 channels, 32 x
32, 32 x 64, the k-split one) against the oracle: tile counts and channels that fill nothing evenly, views
whose output cannot be stored 8 bytes at a time, fp32 output, residual and amax slots."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from aexrt_amd import kernels as K
from aexrt_amd import packing
from tests.helpers import he_weight, nchw_to_nhwc, nhwc_to_nchw, tol_range

pytestmark = pytest.mark.gpu

FP16_TOL = 1e-2

CASES = [
    # n, c, h, w, oc, residual, fp32 output, first channel of x and y in a wider tensor (None: dense)
    (1, 4, 2, 2, 8, False, False, None),         # one tile
    (1, 32, 6, 10, 64, False, False, None),      # 15 tiles
    (3, 36, 8, 22, 70, True, False, None),       # 132 tiles, a second chunk of 4 channels, OC past a block
    (2, 100, 14, 6, 40, False, True, None),
    (1, 64, 34, 32, 64, True, True, (8, 8)),     # slices, 16-byte aligned output
    (1, 64, 12, 12, 38, True, False, (8, 2)),    # output slice of 4-byte alignment, OC % 4 == 2
    (1, 160, 10, 10, 48, False, False, None),    # split k, 5 chunks over 4 waves
    (2, 128, 6, 4, 6, True, False, (0, 1)),      # split k, odd output slice
    (9, 12, 44, 44, 24, False, False, None),     # 4356 tiles x 24 channels: 32 x 32 blocks
    (17, 8, 64, 62, 68, True, False, None),      # 16864 tiles, two channel blocks: 32 x 64
]


@pytest.mark.parametrize("case", CASES)
def test_winograd_sizes(cuda, case):
    import torch

    n, c, h, w, oc, residual, f32, cut = case
    rng = np.random.default_rng(c + oc)
    x = O.round_f16(rng.standard_normal((n, c, h, w)).astype(np.float32))
    wt = he_weight(rng, oc, c, 3)
    b = packing.fp16_round(rng.uniform(-0.1, 0.1, oc).astype(np.float32))
    desc = O.conv_desc(n, c, h, w, oc, 3, 1, 1)
    pc = K.prepare_conv(desc, 40, K.SRC_LAYOUT_WINO_F16, packing.pack_winograd_f2x2_fp16(wt), b, device=cuda)
    x0, y0 = cut or (0, 0)
    xd = torch.zeros((n, h, w, c + 2 * x0), dtype=torch.float16, device=cuda)
    xd[..., x0:x0 + c] = torch.from_numpy(nchw_to_nhwc(x.astype(np.float16))).to(cuda)
    whole = torch.full((n, h, w, oc + 2 * y0), 77.0, dtype=torch.float32 if f32 else torch.float16, device=cuda)
    y = whole[..., y0:y0 + oc]
    r = O.round_f16(rng.standard_normal((n, oc, h, w)).astype(np.float32)) if residual else None
    rd = torch.from_numpy(nchw_to_nhwc(r.astype(np.float16))).to(cuda) if residual else None
    ys = K.new_slots((oc + 15) // 16 * 16, cuda, stripes=4)
    K.conv2d(pc, xd[..., x0:x0 + c], y, flags=K.SILU | (K.RESIDUAL if residual else 0) | (K.OUT_F32 if f32 else 0),
             y_slots=ys, residual=rd)
    torch.cuda.synchronize()
    got = nhwc_to_nchw(y.float().cpu().numpy())
    want = O.winograd_conv(x, O.winograd_weight(wt, to_f16=True), b, desc)
    err, allowed = tol_range(want + r if residual else want, got, FP16_TOL)
    assert err <= allowed, (err, allowed)
    # nothing beside the slice is written; the slots hold the stored maxima
    assert bool((whole[..., :y0] == 77.0).all()) and bool((whole[..., y0 + oc:] == 77.0).all())
    groups = [np.float32(np.abs(got[:, g:g + 16]).max()).view(np.uint32) for g in range(0, oc, 16)]
    np.testing.assert_array_equal(K.slots_max(ys), groups)
