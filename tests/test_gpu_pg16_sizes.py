"""pg16 convs at the edges of their tiles: the NHWC kernels (64-position and window tiles, 1, 2 and 4 channel
subtiles a wave) give the bits of the reference's packed form, whether the strip maxima come as one copy, as
striped slots or as the command's own parts; the command also where its parts do not fit its scratch."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from aexrt_amd import kernels as K
from aexrt_amd import packing

pytestmark = pytest.mark.gpu

CASES = [
    # n, c, h, w, oc, k, stride
    (1, 16, 17, 16, 8, 3, 1),       # one group
    (1, 48, 13, 11, 16, 3, 2),      # 42 positions
    (3, 48, 33, 17, 144, 3, 1),     # short grid of few groups: 64-position tiles
    (2, 128, 31, 33, 64, 3, 1),     # window tiles from 128 channels on
    (1, 112, 31, 33, 64, 3, 1),     # and below them
    (8, 64, 29, 41, 40, 3, 1),      # window tiles by the grid
    (16, 32, 61, 35, 72, 3, 2),
    (2, 688, 9, 10, 272, 3, 1),     # 43 groups: their weights do not fit the window kernel's LDS
    (1, 128, 9, 9, 24, 1, 1),       # 1x1, one subtile
    (9, 80, 40, 41, 48, 1, 1),      # two (groups not a multiple of four)
    (9, 128, 41, 43, 64, 1, 1),     # four
    (5, 2048, 16, 16, 16, 1, 1),    # 128 groups: atomic strips
]


@pytest.mark.parametrize("case", CASES)
def test_nhwc_forms_equal_the_packed_form(cuda, case):
    import torch

    n, c, h, w, oc, k, s = case
    rng = np.random.default_rng(c + oc)
    g = torch.Generator(device="cuda").manual_seed(h)
    x = torch.randn((n, h, w, c), generator=g, device=cuda)
    x = (x * (4.0 ** (torch.arange(c, device=cuda) // 16 % 5 - 2))).half()
    wt = (rng.standard_normal((oc, c, k, k)) / np.sqrt(c * k * k)).astype(np.float32)
    pc = K.prepare_conv(O.conv_desc(n, c, h, w, oc, k, s, k // 2), 51 if k == 1 else 52 if s == 1 else 53,
                        K.SRC_LAYOUT_INT8, packing.pack_conv_int8(wt, fp16_engine=True),
                        rng.uniform(-0.1, 0.1, oc).astype(np.float32), device=cuda)
    oh, ow = (h - 1) // s + 1, (w - 1) // s + 1
    strips = K.amax_strips_nhwc(x)
    flags = K.SILU | K.OUT_F32
    amax = torch.cat([torch.zeros(1, dtype=torch.int32, device=cuda), strips])
    packed = K.quant_pack_nchw(x.permute(0, 3, 1, 2).contiguous(), amax, per_group=True)
    want = torch.empty((n, oc, oh, ow), dtype=torch.float32, device=cuda)
    K.conv2d_int8_pg16(pc, packed, amax, want, flags=flags)
    want = want.permute(0, 2, 3, 1).contiguous().view(torch.int32)

    striped = torch.zeros((5, c // 16), dtype=torch.int32, device=cuda)
    striped[torch.arange(c // 16, device=cuda) % 5, torch.arange(c // 16, device=cuda)] = strips
    for slots in (strips, striped, None):
        y = torch.full((n, oh, ow, oc), 7.0, dtype=torch.float32, device=cuda)
        if slots is None:
            K.conv2d_int8(pc, x, y, flags=flags | K.INT8_PG16)
        else:
            K.conv2d(pc, x, y, flags=flags | K.INT8_PG16, x_slots=slots)
        torch.cuda.synchronize()
        assert torch.equal(y.view(torch.int32), want)
