"""The int8 command's amax in parts: the same outputs, bit for bit, as the conv with the input's 16-channel
amax slots, with the largest element anywhere in the tensor (the first and last chunk, the edges of a
block's share), on dense tensors and channel slices, from one part to all of them, and for zero and
infinite inputs."""
from __future__ import annotations

import numpy as np
import pytest

from aexrt_amd import kernels as K
from aexrt_amd import packing
import oracle as O

pytestmark = pytest.mark.gpu

CASES = [
    # n, c, h, w, slice (channels of the tensor the input is cut from, first channel)
    (1, 16, 16, 16, None),        # the smallest per-tensor command: 512 chunks, one part
    (1, 32, 33, 31, None),        # 4092 chunks: three parts
    (2, 64, 40, 26, None),        # 16640
    (1, 16, 37, 29, (48, 16)),    # a channel slice
    (3, 128, 20, 20, (256, 128)),
    (8, 64, 128, 130, None),      # 1064960 chunks: every part, more than a sweep of them
    (5, 80, 64, 67, (96, 0)),
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("at", ["first", "last", "middle", "zero", "inf"])
def test_int8_command_amax_parts(cuda, case, at):
    import torch

    n, c, h, w, cut = case
    g = torch.Generator(device="cuda").manual_seed(n * c)
    ct, c0 = cut or (c, 0)
    whole = torch.randn((n, h, w, ct), generator=g, device=cuda).half()
    x = whole[..., c0:c0 + c]
    if at == "zero":
        x.zero_()
    else:
        flat = {"first": (0, 0, 0, 0), "last": (n - 1, h - 1, w - 1, c - 1)}.get(at, (n // 2, h // 2, w - 1, c // 2))
        x[flat] = float("inf") if at == "inf" else -37.5
    rng = np.random.default_rng(1)
    wt = (rng.standard_normal((16, c, 1, 1)) / np.sqrt(c)).astype(np.float32)
    desc = O.conv_desc(n, c, h, w, 16, 1, 1, 0)
    pc = K.prepare_conv(desc, 51, K.SRC_LAYOUT_INT8, packing.pack_conv_int8(wt, fp16_engine=True),
                        np.zeros(16, np.float32), device=cuda)
    slots = K.new_slots(c, cuda)
    K.amax_slots(x, slots)
    want = torch.empty((n, h, w, 16), dtype=torch.float16, device=cuda)
    K.conv2d(pc, x, want, x_slots=slots)
    for run in (K.conv2d_int8, K.conv2d_int8_noalloc):
        y = torch.full_like(want, 3.0)
        run(pc, x, y)
        assert torch.equal(y.view(torch.int16), want.view(torch.int16))
