"""The dynamic int8 conv at the edges of its steps and blocks, fp32 output without SiLU bit for bit
against the oracle: channels that do not fill a 64-channel step, one or several steps of the 1x1's
eight, output channels that do not fill a 16-channel tile or a block of four, positions one to a block
and four to a block (with a remainder), and a zero input."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from aexrt_amd import kernels as K
from aexrt_amd import packing
from tests.helpers import nchw_to_nhwc, nhwc_to_nchw

pytestmark = pytest.mark.gpu

CASES = [
    # n, c, h, w, oc, k, s
    (1, 16, 1, 1, 8, 1, 1),
    (1, 16, 3, 2, 8, 3, 1),
    (2, 48, 3, 5, 24, 3, 2),
    (1, 80, 4, 7, 72, 3, 1),       # second step of one 16-channel row
    (1, 528, 2, 3, 40, 1, 1),      # 9 steps: one past a load of eight
    (1, 1104, 1, 1, 16, 1, 1),     # 18: two loads and two over
    (1, 1024, 2, 1, 16, 3, 1),
    (1, 64, 33, 31, 24, 3, 1),     # four positions to a block, 1023 of them
    (3, 32, 37, 19, 136, 1, 1),    # the same, 2109
    (2, 64, 67, 33, 8, 3, 2),      # the same, stride 2
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("zero", [False, True])
def test_dynamic_conv_sizes_bit_exact(cuda, case, zero):
    import torch

    n, c, h, w, oc, k, s = case
    rng = np.random.default_rng(c + oc)
    x = O.round_f16(rng.standard_normal((n, c, h, w)).astype(np.float32) * (0.0 if zero else 3.0))
    wt = (rng.standard_normal((oc, c, k, k)) / np.sqrt(c * k * k)).astype(np.float32)
    b = packing.fp16_round(rng.uniform(-0.1, 0.1, oc).astype(np.float32))
    desc = O.conv_desc(n, c, h, w, oc, k, s, k // 2)
    alg = 51 if k == 1 else (53 if s == 2 else 52)
    pc = K.prepare_conv(desc, alg, K.SRC_LAYOUT_INT8, packing.pack_conv_int8(wt, fp16_engine=True), b, device=cuda)
    _, _, oh, ow = O.out_shape(desc)
    y = torch.full((n, oh, ow, oc), -7.0, dtype=torch.float32, device=cuda)
    ys = K.new_slots(oc, cuda, stripes=4)
    xd = torch.empty((n, h, w, c), dtype=torch.float16, device=cuda)
    xd.copy_(torch.from_numpy(nchw_to_nhwc(x.astype(np.float16))))
    K.conv2d(pc, xd, y, flags=K.INT8_DYNAMIC | K.OUT_F32, y_slots=ys)
    torch.cuda.synchronize()
    qw, ws = O.weight_quant(wt, fp16_round=True)
    got, want = nhwc_to_nchw(y.cpu().numpy()), O.conv_int8_dynamic(x, qw, desc, ws, b, False)
    np.testing.assert_array_equal(got, want)
    groups = [np.float32(np.abs(got[:, g:g + 16]).max()).view(np.uint32) for g in range(0, oc, 16)]
    np.testing.assert_array_equal(K.slots_max(ys), groups)
