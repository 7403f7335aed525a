"""The wave-per-syndrome executor of fused_f32 and fused_f64 against the
workgroup tiles of the same modes, bit for bit (they run the same chain of
operations per entry), where it can go wrong: one row, ragged tiles, every
number of syndromes per wave, listed rows, rows that are all re-checked,
steps with labels summed on one side only, outputs narrower and wider than a
wave, and re-pinned tiles.  Marginals of the hand-made plans against the CPU
oracle at the tolerances of _parity.py / 1e-12.
"""
import numpy as np
import pytest

from _parity import check_f32
from oracle.cexec import OraclePlan
from tensorqec import decoders as D
from tensorqec import lib as L
from tensorqec.codes import CSSTannerGraph, ShorCode, SteaneCode, SurfaceCode
from tensorqec.errors import css_syndrome_rows, iid_error, sample_depolarizing
from tensorqec.planner import Plan

pytestmark = pytest.mark.gpu


def run(torch, hip, S, mode, rows=None):
    n, nout = len(S), 1 << hip.n_out
    dS = torch.from_numpy(np.ascontiguousarray(S)).to("cuda:0")
    mar = torch.full((n, nout), -1.0, dtype=torch.float64, device="cuda:0")
    cls = torch.full((n,), -1, dtype=torch.int32, device="cuda:0")
    tie = torch.full((n,), 7, dtype=torch.uint8, device="cuda:0")
    out = (mar, cls, tie)
    if rows is None:
        hip.decode_device(dS.data_ptr(), n, mode, *(x.data_ptr() for x in out))
    else:
        dl = torch.from_numpy(np.asarray(rows, np.int32)).to("cuda:0")
        dc = torch.tensor([len(rows)], dtype=torch.int32, device="cuda:0")
        hip.decode_list_device(dS.data_ptr(), dl.data_ptr(), dc.data_ptr(), n, mode, *(x.data_ptr() for x in out))
    return [x.cpu().numpy() for x in out] + [hip.last_recheck_count() if mode == "fused_f32" else 0]


def both(torch, hip, S, tiles, rows=None):
    """The wave executor's outputs, equal to the tiles' in both modes."""
    got = {}
    for mode in ("fused_f32", "fused_f64"):
        for m in ("fused_f32", "fused_f64"):
            hip.set_tile(m, 1, 64)
        got[mode] = run(torch, hip, S, mode, rows)
        for m in ("fused_f32", "fused_f64"):
            hip.set_tile(m, *tiles)
        for a, b in zip(got[mode], run(torch, hip, S, mode, rows)):
            assert np.array_equal(a, b), mode
    return got


@pytest.mark.parametrize("code", [SteaneCode(), ShorCode(), SurfaceCode(3, 3), SurfaceCode(5, 5), SurfaceCode(7, 7)], ids=str)
@pytest.mark.parametrize("n", [1, 67, 4999, 20001])
def test_wave_equals_tiles(code, n):
    torch = pytest.importorskip("torch")
    t = CSSTannerGraph.from_code(code)
    em = iid_error(0.03, 0.02, 0.03, t.nq)
    ct = D.compile(D.TNMMAP(), t, em)
    S = css_syndrome_rows(sample_depolarizing(em, seed=n, count=n), t)
    tiles = (8, 128)
    first = run(torch, ct.hip, S, "fused_f32")             # the default choice
    got = both(torch, ct.hip, S, tiles)
    for a, b in zip(first, got["fused_f32"]):
        assert np.array_equal(a, b)
    both(torch, ct.hip, S, tiles, rows=np.arange(n)[::-3])
    if n < 5000:
        ct.hip.set_tolerances(1e-12, 2.0)                  # every row re-checked
        got = both(torch, ct.hip, S, tiles)
        for a, b in zip(got["fused_f32"][:3], got["fused_f64"][:3]):
            assert np.array_equal(a, b)
        assert got["fused_f32"][3] == n


def chain(ra, rb, single, seed):
    """Two evidence-dependent leaves joined by rb labels, ra more labels of
    each kept; then joined to a third with the output's two; `single` labels
    of the first product are summed on its side alone."""
    rng = np.random.default_rng(seed)
    ev = [0, 1, 2]
    a = list(range(10, 10 + ra))
    k = list(range(30, 30 + rb))
    b = list(range(50, 50 + ra))
    o = [70, 71]
    s = a[:single]
    leaves = [[ev[0]] + a + k, [ev[1]] + k + b, [ev[2]] + a[single:] + b + o]
    data = [rng.uniform(0.1, 1.0, 1 << len(x)) for x in leaves]
    return Plan(3, leaves, data, [-1] * 3, [0, 3], [1, 2], [a + b, o], o, 3, {0: 0, 1: 1, 2: 2}), s


@pytest.mark.parametrize("ra,rb,single", [(1, 0, 0), (1, 1, 1), (2, 3, 1), (3, 2, 2), (3, 4, 3), (4, 1, 1), (4, 3, 2)])
def test_wave_single_sided_sums(ra, rb, single):
    torch = pytest.importorskip("torch")
    plan, _ = chain(ra, rb, single, 7 * ra + rb)
    hip = L.HipPlan(plan, tabulate_bits=1)
    S = np.array([[(i >> j) & 1 for j in range(3)] for i in range(8)] * 9, np.uint8)
    got = both(torch, hip, S, (4, 64))
    ref, _, _ = OraclePlan(plan).decode(S)
    m = got["fused_f64"][0]
    assert np.max(np.abs(m - ref) / ref) < 1e-12
    check_f32(got["fused_f32"][0], got["fused_f32"][1], ref, "chain")


def test_autotune_keeps_the_results():
    torch = pytest.importorskip("torch")
    t = CSSTannerGraph.from_code(SurfaceCode(3, 3))
    em = iid_error(0.03, 0.02, 0.03, t.nq)
    ct = D.compile(D.TNMMAP(), t, em)
    S = css_syndrome_rows(sample_depolarizing(em, seed=5, count=3000), t)
    before = run(torch, ct.hip, S, "fused_f32")
    dS = torch.from_numpy(np.ascontiguousarray(S)).to("cuda:0")
    tile, threads = ct.hip.autotune("fused_f32", dS.data_ptr(), len(S))
    for pinned in (False, True):
        if pinned:
            ct.hip.set_tile("fused_f32", tile, threads)
        for a, b in zip(before, run(torch, ct.hip, S, "fused_f32")):
            assert np.array_equal(a, b)
