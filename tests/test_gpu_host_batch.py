"""Host batches: decoding and error-pattern recovery in one call, against the
device-pointer decode and the integer products of css_error_patterns (whole
numbers: equal).  Sizes on both sides of the directly addressed, staged and
unstaged transfers; codes with more than 64 qubits or checks and with two
logical pairs; matrices the one-call path does not take."""
import numpy as np
import pytest

from tensorqec import decoders as D
from tensorqec.codes import CSSTannerGraph, SurfaceCode, ToricCode
from tensorqec.errors import css_syndrome_rows, iid_error, sample_depolarizing

pytestmark = pytest.mark.gpu


def device(torch, ct, S, mode):
    n = len(S)
    dS = torch.from_numpy(np.ascontiguousarray(S)).to("cuda:0")
    out = (torch.empty((n, 1 << ct.hip.n_out), dtype=torch.float64, device="cuda:0"),
           torch.empty(n, dtype=torch.int32, device="cuda:0"), torch.empty(n, dtype=torch.uint8, device="cuda:0"))
    ct.hip.decode_device(dS.data_ptr(), n, mode, *(x.data_ptr() for x in out))
    return [x.cpu().numpy() for x in out] + [ct.hip.last_recheck_count()]


def same(torch, ct, S, mode, want_marginals=True):
    r = D.decode_batch(ct, S, mode=mode, want_marginals=want_marginals)
    count = ct.hip.last_recheck_count()
    mar, cls, tie, ref_count = device(torch, ct, S, mode)
    assert (r.marginals is None) if not want_marginals else np.array_equal(r.marginals, mar)
    assert np.array_equal(r.classes, cls) and np.array_equal(r.ties, tie) and count == ref_count
    ep = D.css_error_patterns(ct, S, cls)
    for a, b in ((r.error_patterns.xerror, ep.xerror), (r.error_patterns.zerror, ep.zerror)):
        assert a.dtype == b.dtype and a.shape == b.shape and np.array_equal(a, b)


def compiled(code, greedy=False):
    t = CSSTannerGraph.from_code(code)
    em = iid_error(0.02, 0.01, 0.03, t.nq)
    return t, em, D.compile(D.TNMMAP(optimizer=D.GreedyMethod()) if greedy else D.TNMMAP(), t, em)


@pytest.mark.parametrize("code,sizes", [(SurfaceCode(3, 3), [1, 2, 63, 4097, 200001]), (SurfaceCode(5, 5), [1, 1000]),
                                        (SurfaceCode(9, 9), [1, 65]), (ToricCode(2, 2), [1, 130]),
                                        (ToricCode(3, 3), [1, 100])], ids=str)
def test_one_call(code, sizes):
    torch = pytest.importorskip("torch")
    t, em, ct = compiled(code)
    mode = "fused_f32" if ct.hip.stats()["fused_lds_entries"] < 20000 else "spec_f32"
    for n in sizes:
        S = css_syndrome_rows(sample_depolarizing(em, seed=n, count=n), t)
        for want in (True, False):
            same(torch, ct, S, mode, want)
    r = D.decode_batch(ct, np.zeros((0, t.ns), np.uint8))
    assert r.classes.shape == (0,) and r.error_patterns.xerror.shape == (0, t.nq)


def test_other_matrices():
    torch = pytest.importorskip("torch")
    t, em, ct = compiled(SurfaceCode(3, 3))
    S = css_syndrome_rows(sample_depolarizing(em, seed=3, count=200), t)
    ct.pure_x = np.asfortranarray(ct.pure_x)
    same(torch, ct, S, "fused_f32")
    ct.lx = ct.lx * np.uint8(3)                       # not 0/1: the integer products decide
    same(torch, ct, S, "fused_f32")
    ct.lx = (ct.lx // np.uint8(3)).astype(np.int64)
    ct.pure_z = ct.pure_z.astype(np.int64)
    ref = D.css_error_patterns(ct, S, device(torch, ct, S, "fused_f32")[1])
    got = D.decode_batch(ct, S).error_patterns
    assert np.array_equal(got.xerror, ref.xerror) and np.array_equal(got.zerror, ref.zerror)
