"""The fp16 table of V centroids that is laid out once follows the centroids (no GPU)."""
import copy
import pickle

import pytest
import torch

from blockgtq_amd.v_quantize_gpu import PolarQuantGPU


def _follows(q):
    assert q.v_lut.dtype == torch.float16 and torch.equal(q.v_lut, q.centroids.half())


@pytest.mark.parametrize("bits", [1, 3, 4])
def test_table_follows_the_centroids(bits):
    q = PolarQuantGPU(128, bits)
    _follows(q)
    assert q.v_lut is q.v_lut
    q.centroids.mul_(2)
    _follows(q)
    q.v_lut.zero_()                                   # (the table is the caller's to change as before)
    _follows(q)
    q.centroids = q.centroids + 1
    _follows(q)
    for other in (copy.deepcopy(q), pickle.loads(pickle.dumps(q))):
        other.centroids.add_(1)
        _follows(other)
    del q.__dict__['_lut']                            # (an object that was saved without the table)
    _follows(q)


def test_tensors_without_versions():
    q = PolarQuantGPU(128, 3)
    with torch.inference_mode():
        _follows(q)
        made = PolarQuantGPU(128, 3)
        _follows(made)
    _follows(made)
    with torch.inference_mode():
        made.centroids.mul_(2)
    _follows(made)
