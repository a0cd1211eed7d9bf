"""Which weights a packed copy counts for (``models/projection.py``)."""
import pytest
import torch

from omnia_amd import ops
from omnia_amd.models.projection import Projections, packed_copy, version


@pytest.mark.parametrize("inference", [False, True])
def test_a_copy_counts_while_the_weight_is_what_was_copied(inference, monkeypatch):
    """Weights made in inference mode have no version to compare: their copies count."""
    with torch.inference_mode(inference):
        w = torch.randn(32, 64).to(torch.bfloat16)
    copy, x = w.clone(), torch.randn(200, 64).to(torch.bfloat16)
    m = Projections()
    m._streams = {w.data_ptr(): (w, version(w), copy)}
    m._packed = {(w.data_ptr(), 128, 0): (w, version(w), copy)}
    monkeypatch.setattr(ops, "tgemm", lambda mode, x, w, *a: w)
    monkeypatch.setattr(ops, "wgemm", lambda mode, x, w, *a, out=None: w)

    def read(w):
        tile = m._wgemm(0, x, w, 1, 128, -1)
        assert (tile is copy) == (packed_copy(m, w) is copy)
        return tile

    assert read(w) is copy
    half = w[:16]
    assert read(half) is half  # at its address, of another shape
    square = w.view(64, 32).t()
    assert square.shape == w.shape and read(square) is square  # of other strides
    if not inference:
        w.neg_()
        assert read(w) is w
