"""3x3 convs without a measured tile: whatever tile the estimated times pick, int8 gives the implicit
GEMM's outputs, accumulators and amax slots bit for bit, and fp16 stays within fp32 accumulation of a
float64 conv - over small and large maps, odd sizes, both strides, channel slices, a residual, fp32
output, and with a tile forced on the implicit GEMM."""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from aexrt_amd import kernels as K
from aexrt_amd import packing

pytestmark = pytest.mark.gpu

SHAPES = [
    # n, c, h, w, oc, stride, flags, slice of the input, of the output (channels of the tensor, first channel)
    (1, 16, 1, 1, 8, 1, K.SILU, None, None),
    (1, 16, 2, 3, 16, 2, K.SILU, None, None),
    (1, 64, 5, 5, 64, 1, K.SILU, None, None),
    (7, 16, 26, 26, 224, 1, K.SILU, None, None),
    (2, 256, 40, 40, 256, 1, K.SILU, None, None),
    (1, 512, 20, 20, 512, 1, K.SILU, None, None),
    (4, 64, 81, 79, 128, 2, K.SILU, None, None),
    (16, 144, 67, 73, 32, 1, K.SILU, None, None),
    (9, 208, 7, 6, 96, 1, 0, None, None),
    (3, 320, 51, 47, 112, 2, K.SILU, (336, 16), (128, 8)),
    (2, 96, 27, 35, 48, 1, K.SILU | K.RESIDUAL, None, None),
    (2, 128, 33, 31, 80, 1, K.SILU | K.OUT_F32, (256, 128), None),
]


def _conv(shape, int8, cuda):
    import torch

    n, c, h, w, oc, s, flags, xs, ys = shape
    g = torch.Generator(device="cuda").manual_seed(c + oc + h)
    ct, c0 = xs or (c, 0)
    x = torch.randn((n, h, w, ct), generator=g, device=cuda).half()[..., c0:c0 + c]
    rng = np.random.default_rng(oc)
    wt = (rng.standard_normal((oc, c, 3, 3)) / np.sqrt(9 * c)).astype(np.float32)
    b = rng.uniform(-0.1, 0.1, oc).astype(np.float32)
    d = O.conv_desc(n, c, h, w, oc, 3, s, 1)
    if int8:
        pc = K.prepare_conv(d, 52 if s == 1 else 53, K.SRC_LAYOUT_INT8, packing.pack_conv_int8(wt, fp16_engine=True), b, device=cuda)
    else:
        pc = K.prepare_conv(d, 5, K.SRC_RAW_F32, wt, b, device=cuda)
    return pc, x, wt, b


def _run(shape, pc, x, int8, cuda, acc_on=False):
    import torch

    n, c, h, w, oc, s, flags, xs, ys = shape
    oh, ow = (h - 1) // s + 1, (w - 1) // s + 1
    yt, y0 = ys or (oc, 0)
    slots = None
    if int8:
        slots = K.new_slots(c, cuda)
        K.amax_slots(x, slots)
    g = torch.Generator(device="cuda").manual_seed(oc)
    res = torch.randn((n, oh, ow, oc), generator=g, device=cuda).half() if flags & K.RESIDUAL else None
    whole = torch.full((n, oh, ow, yt), 5.0, dtype=torch.float32 if flags & K.OUT_F32 else torch.float16, device=cuda)
    yslots = K.new_slots((oc + 15) // 16 * 16, cuda, stripes=4)
    acc = torch.full((n * oh * ow, oc), -1, dtype=torch.int32, device=cuda) if acc_on else None
    K.conv2d(pc, x, whole[..., y0:y0 + oc], flags=flags, x_slots=slots, y_slots=yslots, residual=res, acc_out=acc)
    torch.cuda.synchronize()
    return whole, K.slots_max(yslots), acc, res


@pytest.mark.parametrize("acc_on", [False, True])
@pytest.mark.parametrize("shape", SHAPES)
def test_int8_equals_the_implicit_gemm(cuda, shape, acc_on):
    import torch

    pc, x, _, _ = _conv(shape, True, cuda)
    whole, slots, acc, _ = _run(shape, pc, x, True, cuda, acc_on)
    others = []
    try:
        K.set_conv_tile(1, 1)  # the window kernels still go first
        others.append(_run(shape, pc, x, True, cuda, acc_on))
        K.set_conv3x3_halo(K.HALO_OFF)
        others.append(_run(shape, pc, x, True, cuda, acc_on))
    finally:
        K.set_conv_tile()
        K.set_conv3x3_halo()
    as_int = torch.int32 if whole.dtype == torch.float32 else torch.int16
    for whole2, slots2, acc2, _ in others:
        assert torch.equal(whole.view(as_int), whole2.view(as_int))
        np.testing.assert_array_equal(slots, slots2)
        if acc_on:
            assert torch.equal(acc, acc2)


@pytest.mark.parametrize("shape", SHAPES + [(3, 8, 11, 13, 24, 1, K.SILU, None, None),
                                            (2, 184, 45, 52, 72, 2, K.SILU, None, None)])
def test_fp16_within_fp32_accumulation(cuda, shape):
    import torch
    import torch.nn.functional as F

    n, c, h, w, oc, s, flags, xs, ys = shape
    pc, x, wt, b = _conv(shape, False, cuda)
    whole, _, _, res = _run(shape, pc, x, False, cuda)
    y0 = (ys or (oc, 0))[1]
    xd = x.cpu().double().permute(0, 3, 1, 2)
    wd = torch.from_numpy(wt.astype(np.float16)).double()
    bd = torch.from_numpy(b).double()
    ref = F.conv2d(xd, wd, bd, stride=s, padding=1)
    mag = F.conv2d(xd.abs(), wd.abs(), bd.abs(), stride=s, padding=1)
    # any order of the 9 c products and the bias in fp32
    bound = (9 * c + 1) * 2.0 ** -24 * mag
    if flags & K.SILU:
        ref = ref * torch.sigmoid(ref)
        bound = 1.1 * bound + 2.0 ** -20 * mag.clamp(min=1.0)  # slope of SiLU below 1.1; its fp32 exp
    if res is not None:
        ref = ref + res.cpu().double().permute(0, 3, 1, 2)
    if not flags & K.OUT_F32:
        bound = bound + 2.0 ** -11 * ref.abs() + 2.0 ** -25
        if res is not None:
            bound = bound + 2.0 ** -11 * (ref.abs() + 1.0)  # rounded before and after the residual
    got = whole[..., y0:y0 + oc].cpu().double().permute(0, 3, 1, 2)
    worst = ((got - ref).abs() - bound).max().item()
    assert worst <= 0.0, worst
    if ys:
        untouched = torch.cat([whole[..., :y0], whole[..., y0 + oc:]], -1)
        assert bool((untouched == 5.0).all())
