"""The fp16 table of V centroids is what the centroids are when it is read, and its reader's own."""
import copy
import pickle

import pytest
import torch

from blockgtq_amd.v_quantize_gpu import PolarQuantGPU


def _follows(q):
    assert q.v_lut.dtype == torch.float16 and torch.equal(q.v_lut, q.centroids.half())


@pytest.mark.parametrize("bits", [1, 3, 4])
def test_table_follows_the_centroids_however_they_are_changed(bits):
    q = PolarQuantGPU(128, bits)
    _follows(q)
    q.centroids.mul_(2)
    _follows(q)
    q.centroids.data.mul_(2)                          # (counted by no version)
    _follows(q)
    q.centroids.numpy()[:] *= 2
    _follows(q)
    q.centroids.data = q.centroids.data + 1
    _follows(q)
    q.centroids = q.centroids + 1
    _follows(q)
    with torch.inference_mode():
        q.centroids.add_(1)
        _follows(q)
    for other in (copy.deepcopy(q), pickle.loads(pickle.dumps(q))):
        other.centroids.data.add_(1)
        _follows(other)


def test_each_reader_has_a_table_of_its_own():
    q = PolarQuantGPU(128, 3)
    mine, theirs = q.v_lut, q.v_lut
    theirs.zero_()
    assert torch.equal(mine, q.centroids.half())
    assert q.centroids.untyped_storage().nbytes() == q.centroids.nbytes       # (and the centroids share theirs with none)


@pytest.mark.gpu
def test_table_read_under_capture():
    """Replays read the centroids as they are then, and what was only recorded is nobody else's table."""
    q = PolarQuantGPU(128, 3, device="cuda:0")
    _follows(q)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        q.centroids = q.centroids * 2
        side.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            table = q.v_lut
    _follows(q)                                       # before any replay
    for _ in range(3):
        q.centroids.data.mul_(1.5)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(table, q.centroids.half())
        _follows(q)
