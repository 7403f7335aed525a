"""The sampler's blocks of 64 samples where they end: single samples, ragged
last blocks, outputs at odd addresses (byte stores), a model whose masks
outgrow the LDS (the thread-per-sample kernel), and the logical-error loop on
such batches.  Bit-identical to the host sampler, as everywhere.
"""
import numpy as np
import pytest

from tensorqec import decoders as D
from tensorqec import lib as L
from tensorqec.codes import CSSTannerGraph, SurfaceCode
from tensorqec.errors import (IndependentFlipError, check_logical_error, css_syndrome_rows, iid_error,
                              sample_depolarizing, sample_flips)
from tensorqec.gf2 import logical_operator

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000])
@pytest.mark.parametrize("shift", [0, 1])
def test_css_sampler_blocks(n, shift):
    torch = pytest.importorskip("torch")
    t = CSSTannerGraph.from_code(SurfaceCode(3, 5))
    em = iid_error(0.1, 0.05, 0.08, t.nq)
    lx, lz = logical_operator(t)
    first = (1 << 32) - 40   # the counter's high word changes inside a block
    syn, err = (torch.full((n * w + 8,), 9, dtype=torch.uint8, device="cuda:0") for w in (t.ns, 2 * t.nq))
    cls = torch.full((n + 1,), -1, dtype=torch.int32, device="cuda:0")
    L.HipSampler.css(t, em, lx, lz).sample(77, first, n, syn.data_ptr() + shift, cls.data_ptr(), err.data_ptr() + shift)
    torch.cuda.synchronize()
    ep = sample_depolarizing(em, 77, n, first=first)
    want = np.concatenate([ep.xerror, ep.zerror], axis=1)
    got = err.cpu().numpy()
    assert np.array_equal(got[shift:shift + n * 2 * t.nq].reshape(n, -1), want)
    got_s = syn.cpu().numpy()
    assert np.array_equal(got_s[shift:shift + n * t.ns].reshape(n, -1), css_syndrome_rows(ep, t))
    for a, w in ((got, 2 * t.nq), (got_s, t.ns)):   # nothing beyond the rows
        assert (a[:shift] == 9).all() and (a[shift + n * w:] == 9).all()
    k = lx.shape[0]
    bits = np.concatenate([ep.zerror @ lx.T % 2, ep.xerror @ lz.T % 2], axis=1)
    assert np.array_equal(cls.cpu().numpy()[:n], (bits << np.arange(2 * k)).sum(axis=1)) and int(cls[n]) == -1


@pytest.mark.parametrize("nm", [5, 7000, 8000])
def test_flip_sampler_sizes(nm):
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(nm)
    p = rng.uniform(0, 0.01, nm)
    p[0], p[-1] = 0.0, 1.0
    Dm, Lm = (rng.random((13, nm)) < 0.1).astype(np.uint8), (rng.random((2, nm)) < 0.1).astype(np.uint8)
    n = 70
    syn = torch.empty((n, 13), dtype=torch.uint8, device="cuda:0")
    err = torch.empty((n, nm), dtype=torch.uint8, device="cuda:0")
    cls = torch.empty(n, dtype=torch.int32, device="cuda:0")
    L.HipSampler.flips(p, Dm, Lm).sample(3, 5, n, syn.data_ptr(), cls.data_ptr(), err.data_ptr())
    torch.cuda.synchronize()
    e = sample_flips(IndependentFlipError(p), 3, n, 5)
    assert np.array_equal(err.cpu().numpy(), e)
    assert np.array_equal(syn.cpu().numpy(), e.astype(np.int64) @ Dm.T % 2)
    assert np.array_equal(cls.cpu().numpy(), (e.astype(np.int64) @ Lm.T % 2) @ np.array([1, 2]))


@pytest.mark.parametrize("n,batch", [(1, 64), (130, 100), (1000, 1 << 16)])
def test_ler_loop_ragged(n, batch):
    pytest.importorskip("torch")
    t = CSSTannerGraph.from_code(SurfaceCode(3, 3))
    em = iid_error(0.05, 0.04, 0.03, t.nq)
    ct = D.compile(D.TNMMAP(mode="spec_f32"), t, em)
    ler = L.HipLER(ct.hip, L.HipSampler.css(t, em, ct.lx, ct.lz),
                   L.HipRecovery.css(t, ct.pure_x, ct.pure_z, ct.lx, ct.lz), batch=batch)
    got = ler.run("spec_f32", 11, 0, n)
    ep = sample_depolarizing(em, 11, n)
    r = D.decode_batch(ct, css_syndrome_rows(ep, t), mode="spec_f32")
    assert got["logical_errors"] == int(check_logical_error(ep, r.error_patterns, ct.lx, ct.lz).sum())
    assert got["inconsistent"] == 0 and got["samples"] == n
