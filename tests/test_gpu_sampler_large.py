"""Sampling in one call more samples than one launch takes (a grid holds fewer
than 2^32 work-items): every output around the edges of the launches, at the
start and at the end, bit-identical to the host sampler."""
import numpy as np
import pytest

from tensorqec import lib as L
from tensorqec.errors import IndependentFlipError, sample_flips

pytestmark = pytest.mark.gpu


def test_samples_of_several_launches():
    torch = pytest.importorskip("torch")
    p = np.array([0.3, 0.05, 0.5])
    Dm, Lm = np.array([[1, 0, 1]], np.uint8), np.array([[0, 1, 1]], np.uint8)
    n, first = (1 << 30) + 65, 7
    syn = torch.full((n, 1), 9, dtype=torch.uint8, device="cuda:0")
    err = torch.full((n, 3), 9, dtype=torch.uint8, device="cuda:0")
    cls = torch.full((n,), -1, dtype=torch.int32, device="cuda:0")
    L.HipSampler.flips(p, Dm, Lm).sample(21, first, n, syn.data_ptr(), cls.data_ptr(), err.data_ptr())
    torch.cuda.synchronize()
    for at in (0, (1 << 29) - 64, (1 << 30) - 64, n - 128):
        e = sample_flips(IndependentFlipError(p), 21, 128, first + at).astype(np.int64)
        assert np.array_equal(err[at:at + 128].cpu().numpy(), e)
        assert np.array_equal(syn[at:at + 128].cpu().numpy(), e @ Dm.T % 2)
        assert np.array_equal(cls[at:at + 128].cpu().numpy(), (e @ Lm.T % 2)[:, 0])
    assert int(syn.max()) == 1 and int(cls.min()) == 0      # every row was written
