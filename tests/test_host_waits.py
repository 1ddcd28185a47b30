"""Host side of the counts the GPU hands over: gsplat_wait_count, and
intersect_tile's emission queued for the last count of the same shape
(Intersect.cpp:104-122 reads the count between its two stages)."""

import ctypes

import pytest
import torch

from gsplat_amd import _lib
from tests._util import DEV


def test_wait_count_returns_a_written_word_and_refuses_null():
    word = ctypes.c_int64(7)
    out = ctypes.c_int64(-5)
    _lib.call("gsplat_wait_count", ctypes.addressof(word), ctypes.addressof(out), None)
    assert out.value == 7
    with pytest.raises(RuntimeError, match="NULL"):
        _lib.call("gsplat_wait_count", None, ctypes.addressof(out), None)


@pytest.mark.gpu
def test_wait_count_on_a_drained_stream_is_an_error():
    word = _lib.host_count()
    torch.zeros(8, device=DEV).add_(1)
    with pytest.raises(RuntimeError, match="nothing queued"):
        _lib.wait_count(word, torch.cuda.current_stream().cuda_stream)


@pytest.mark.gpu
def test_dense_intersection_queued_for_the_last_count():
    """The same shape four times: first with the exact stage, then queued with
    room, with too little (the exact stage again) and with more than enough;
    each equals the exact stage of a shape not seen before."""
    from gsplat_amd.cuda import _ops
    g = torch.Generator().manual_seed(3)
    n, tw, th = 4000, 20, 15
    m2 = (torch.rand(1, n, 2, generator=g) * torch.tensor([320.0, 240.0])).to(DEV)
    dep = torch.rand(1, n, generator=g).to(DEV) + 0.5
    saved = dict(_ops._ISECT_SHAPES)
    try:
        for radius in (6, 7, 40, 3):
            rad = torch.full((1, n, 2), radius, dtype=torch.int32, device=DEV)
            args = (m2, rad, dep, None, None, None, None, 1, 16, tw, th, True, False)
            got = _ops.intersect_tile(*args)
            kept = dict(_ops._ISECT_SHAPES)
            _ops._ISECT_SHAPES.clear()
            want = _ops.intersect_tile(*args)
            _ops._ISECT_SHAPES.clear()
            _ops._ISECT_SHAPES.update(kept)
            for a, b in zip(got, want):
                assert a.shape == b.shape and torch.equal(a, b), radius
    finally:
        _ops._ISECT_SHAPES.clear()
        _ops._ISECT_SHAPES.update(saved)
