"""int8 1x1 convs without a measured tile: the kernel the rule picks gives the implicit GEMM's outputs,
accumulators and amax slots bit for bit, around the rule's lines (positions and channel tiles about 192
and 640, 256 channels) and over the views it accepts (channel slices, fp32 output, no SiLU); residual
convs and a tile forced on the implicit GEMM stay there."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from aexrt_amd import kernels as K
from aexrt_amd import packing

pytestmark = pytest.mark.gpu

CASES = [
    # n, c, h, w, oc, flags, slice of the input, of the output (channels of the tensor, first channel)
    (1, 16, 1, 1, 8, K.SILU, None, None),
    (1, 48, 7, 9, 40, K.SILU, None, None),                  # 63 positions
    (1, 64, 5, 13, 24, K.SILU, (128, 64), (48, 16)),        # 65, slices on both sides
    (2, 128, 78, 78, 128, 0, None, None),                   # 191 tiles of 8 channel subtiles, no SiLU
    (2, 128, 79, 78, 128, K.SILU | K.OUT_F32, None, None),  # 193, fp32 output
    (3, 256, 37, 41, 96, K.SILU, None, None),
    (3, 272, 37, 41, 96, K.SILU, (288, 16), None),
    (8, 304, 71, 72, 16, K.SILU, None, None),               # 640 tiles past 256 channels
    (8, 304, 73, 72, 16, K.SILU, None, None),               # 657
    (2, 512, 10, 10, 264, K.SILU, None, (272, 0)),
    (2, 64, 20, 20, 64, K.SILU | K.RESIDUAL, None, None),
]


def _run(case, cuda, acc_on):
    import torch

    n, c, h, w, oc, flags, xs, ys = case
    g = torch.Generator(device="cuda").manual_seed(c + oc)
    ct, c0 = xs or (c, 0)
    yt, y0 = ys or (oc, 0)
    x = torch.randn((n, h, w, ct), generator=g, device=cuda).half()[..., c0:c0 + c]
    rng = np.random.default_rng(oc)
    wt = (rng.standard_normal((oc, c, 1, 1)) / np.sqrt(c)).astype(np.float32)
    pc = K.prepare_conv(O.conv_desc(n, c, h, w, oc, 1, 1, 0), 51, K.SRC_LAYOUT_INT8,
                        packing.pack_conv_int8(wt, fp16_engine=True),
                        rng.uniform(-0.1, 0.1, oc).astype(np.float32), device=cuda)
    slots = K.new_slots(c, cuda)
    K.amax_slots(x, slots)
    res = torch.randn((n, h, w, oc), generator=g, device=cuda).half() if flags & K.RESIDUAL else None
    whole = torch.full((n, h, w, yt), 5.0, dtype=torch.float32 if flags & K.OUT_F32 else torch.float16, device=cuda)
    yslots = K.new_slots((oc + 15) // 16 * 16, cuda, stripes=4)
    acc = torch.full((n * h * w, oc), -1, dtype=torch.int32, device=cuda) if acc_on else None
    K.conv2d(pc, x, whole[..., y0:y0 + oc], flags=flags, x_slots=slots, y_slots=yslots, residual=res, acc_out=acc)
    torch.cuda.synchronize()
    return whole, K.slots_max(yslots), acc


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("acc_on", [False, True])
def test_rule_equals_the_implicit_gemm(cuda, case, acc_on):
    import torch

    whole, slots, acc = _run(case, cuda, acc_on)
    K.set_conv_tile(1, 1)  # every launch on the implicit GEMM
    try:
        whole2, slots2, acc2 = _run(case, cuda, acc_on)
    finally:
        K.set_conv_tile()
    as_int = torch.int32 if whole.dtype == torch.float32 else torch.int16
    assert torch.equal(whole.view(as_int), whole2.view(as_int))
    np.testing.assert_array_equal(slots, slots2)
    if acc_on:
        assert torch.equal(acc, acc2)
