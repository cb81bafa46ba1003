"""The two-launch postprocess at the edges of its blocks, against the oracle bit for bit.

Anchors around the 64 of a score block, classes around its four quarters and 20-class steps, channels
first and last (rows read 16 bytes at a time or not), saturated and far negative logits (equal
sigmoids: the first class wins), few and many candidates per select block, several streams at once,
and a launch recorded into a graph (which takes the single-block kernel).
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from aexrt_amd import kernels as K

pytestmark = pytest.mark.gpu

# (levels, classes, layout, conf, iou, max candidates, max detections, logit scale, logit shift)
CASES = [
    ([(1, 1, 8.0)], 1, 1, 0.25, 0.45, 1, 1, 2.0, 1.0),
    ([(7, 9, 8.0)], 3, 1, 0.25, 0.45, 16, 5, 2.0, 0.0),
    ([(8, 8, 8.0)], 4, 2, 0.25, 0.45, 17, 100, 2.0, 0.0),
    ([(5, 13, 8.0)], 5, 2, 0.25, 0.45, 512, 100, 2.0, 0.0),
    ([(40, 40, 8.0), (20, 20, 16.0), (10, 10, 32.0)], 80, 2, 0.5, 0.45, 512, 100, 2.0, -1.0),
    ([(40, 40, 8.0), (20, 20, 16.0), (10, 10, 32.0)], 81, 1, 0.5, 0.45, 2048, 300, 2.0, -1.0),
    ([(80, 80, 8.0), (40, 40, 16.0), (20, 20, 32.0)], 16, 2, 0.6, 0.3, 513, 600, 1.0, 0.0),
    ([(20, 20, 8.0), (10, 10, 16.0)], 91, 1, 0.3, 0.0, 300, 300, 30.0, 10.0),   # most sigmoids equal 1
    ([(20, 20, 8.0)], 33, 2, 0.0, 0.9, 300, 300, 60.0, -120.0),                 # and 0, all passing
]


def _head(case, seed):
    levels, classes, layout, *_, scale, shift = case
    a = sum(h * w for h, w, _ in levels)
    rng = np.random.default_rng(seed)
    head = rng.normal(0, 2, (64 + classes, a)).astype(np.float32)
    head[64:] = (head[64:] / 2 * scale + shift).astype(np.float32)
    return np.ascontiguousarray(head.T) if layout == 2 else head


def _want(case, host):
    levels, classes, layout, conf, iou, mc, md, *_ = case
    return O.yolo_dfl_decode_nms_topk(host, levels, classes=classes, layout=layout, conf=conf, iou=iou,
                                      max_candidates=mc, max_detections=md)


def _run(case, dev, **more):
    levels, classes, layout, conf, iou, mc, md, *_ = case
    return K.yolo_dfl_decode_nms_topk(dev, levels, classes=classes, layout=layout, conf=conf, iou=iou,
                                      max_candidates=mc, max_detections=md, **more)


def _equal(got, want):
    got = got.cpu().numpy()
    assert got.shape == want.shape
    np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("case", CASES)
def test_dfl_post_sizes_bit_exact(cuda, case):
    import torch

    host = _head(case, 5)
    _equal(_run(case, torch.from_numpy(host).to(cuda)), _want(case, host))


def test_post_on_more_streams_than_workspaces(cuda):
    """Calls in flight on eight streams at once, twice round: each gets its own result."""
    import ctypes

    import torch

    from aexrt_amd import _lib

    case = CASES[4]
    levels, classes, layout, conf, iou, mc, md, *_ = case
    hosts = [_head(case, 20 + i) for i in range(8)]
    devs = [torch.from_numpy(h).to(cuda) for h in hosts]
    streams = [torch.cuda.Stream() for _ in hosts]
    dets = torch.zeros((16, md, 6), device=cuda)
    counts = torch.zeros(16, dtype=torch.int32, device=cuda)
    hw = (ctypes.c_uint32 * 6)(*[v for h, w, _ in levels for v in (h, w)])
    st = (ctypes.c_float * 3)(*[s for _, _, s in levels])
    torch.cuda.synchronize()
    for turn in range(2):
        for i, (d, s) in enumerate(zip(devs, streams)):
            k = 8 * turn + i
            _lib.check(_lib.lib().aexrt_hip_yolo_dfl_decode_nms_topk(
                d.data_ptr(), layout, 3, hw, st, classes, conf, iou, mc, md, dets[k].data_ptr(),
                counts[k:k + 1].data_ptr(), ctypes.c_void_p(s.cuda_stream)), "yolo_dfl_decode_nms_topk")
    torch.cuda.synchronize()
    for k in range(16):
        _equal(dets[k, : int(counts[k])], _want(case, hosts[k % 8]))


def test_post_recorded_into_a_graph(cuda):
    import ctypes

    import torch

    from aexrt_amd import _lib

    case = CASES[4]
    levels, classes, layout, conf, iou, mc, md, *_ = case
    dev = torch.zeros_like(torch.from_numpy(_head(case, 0))).to(cuda)
    dets = torch.zeros((md, 6), device=cuda)
    count = torch.zeros(1, dtype=torch.int32, device=cuda)
    hw = (ctypes.c_uint32 * 6)(*[v for h, w, _ in levels for v in (h, w)])
    st = (ctypes.c_float * 3)(*[s for _, _, s in levels])
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        _lib.check(_lib.lib().aexrt_hip_yolo_dfl_decode_nms_topk(
            dev.data_ptr(), layout, 3, hw, st, classes, conf, iou, mc, md, dets.data_ptr(), count.data_ptr(),
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "yolo_dfl_decode_nms_topk")
    for seed in (1, 2, 3):
        host = _head(case, seed)
        dev.copy_(torch.from_numpy(host))
        graph.replay()
        torch.cuda.synchronize()
        _equal(dets[: int(count)], _want(case, host))
        _equal(_run(case, dev), _want(case, host))
