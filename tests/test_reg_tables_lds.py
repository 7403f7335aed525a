"""Register-resident kernels with their tables in LDS: the inline FP64
re-check takes what the tables leave of a CU's 160 KB, fewer rows at a time
with their slices staged, then without, then the separate kernel; what the
tables alone do not leave room for is refused, and tuning goes past it."""
import os

import numpy as np
import pytest

from _parity import check_f32, check_f64
from oracle.cexec import OraclePlan
from tensorqec import lib as L
from tensorqec.planner import Plan
from test_host_paths_cpu import run, stub  # noqa: F401  (fixture)


def plan(ev):
    """Five leaves (or fewer), each chosen by so many syndrome bits: 2^9, 2^9,
    2^6, 4 and 4 FP32 entries for each of their patterns."""
    rng = np.random.default_rng(1)
    a, k, b, o = list(range(100, 104)), list(range(110, 115)), list(range(120, 124)), [130, 131]
    leaves, n = [], 0
    for m, labels in zip(ev, [a + k, k + b, a + o, o, o]):
        leaves.append(list(range(n, n + m)) + labels)
        n += m
    q = len(leaves)
    lhs, rhs, outs = [0] + [q + i for i in range(q - 2)], list(range(1, q)), [a + b] + [o] * (q - 2)
    return Plan(q, leaves, [rng.uniform(0.1, 1.0, 1 << len(x)) for x in leaves], [-1] * q, lhs, rhs, outs, o, n,
                {i: i for i in range(n)})


# KB of tables: 69, 133, 145, 152, 158 and 160
EVIDENCE = [[5, 1, 1], [6, 1, 1], [6, 3, 1], [6, 3, 5], [6, 3, 5, 8, 7], [6, 3, 5, 8, 8]]


@pytest.mark.parametrize("ev", EVIDENCE, ids=str)
def test_lds_of_a_workgroup(stub, ev):  # noqa: F811
    _, calls = run(stub, """
sys.path[:0] = [%r]
from test_reg_tables_lds import plan
hip = L.HipPlan(plan(%r), tabulate_bits=0)
S = np.zeros((3, hip.n_syn), np.uint8)
for threads in (64, 128, 256):
    try:
        hip.set_spec(threads // 4, threads, True, reg=True)
        hip.decode(S, "spec_f32")
    except L.TqecError as e:
        assert "does not fit in LDS" in str(e), str(e)
        print("stub refused", file=sys.stderr, flush=True)
if %r:
    hip.autotune("spec_f32", S.ctypes.data, 3)
""" % (os.path.dirname(os.path.abspath(__file__)), ev, ev == EVIDENCE[3]))
    assert calls.count("refused") == (3 if ev[3:] == [8, 8] else 0)
    assert all(int(c.split()[1]) <= 160 * 1024 for c in calls if c.startswith("lds "))


@pytest.mark.gpu
@pytest.mark.parametrize("ev", EVIDENCE[:-1], ids=str)
def test_results_vs_oracle(ev):
    torch = pytest.importorskip("torch")
    p = plan(ev)
    S = np.random.default_rng(2).integers(0, 2, (200, sum(ev)), dtype=np.uint8)
    ref, _, _ = OraclePlan(p).decode(S)
    dS = torch.from_numpy(S).to("cuda:0")
    h = L.HipPlan(p, tabulate_bits=0)
    for threads in (64, 128, 256):
        h.set_spec(threads // 4, threads, True, 0, reg=True)
        for every in (False, True):                 # in FP32, all rows re-checked in FP64
            h.set_tolerances(1e-12, 2.0 if every else 1e-4)
            mar = torch.full((len(S), 4), -1.0, dtype=torch.float64, device="cuda:0")
            cls = torch.full((len(S),), -1, dtype=torch.int32, device="cuda:0")
            tie = torch.full((len(S),), 7, dtype=torch.uint8, device="cuda:0")
            h.decode_device(dS.data_ptr(), len(S), "spec_f32", mar.data_ptr(), cls.data_ptr(), tie.data_ptr())
            mar, cls, tie = mar.cpu().numpy(), cls.cpu().numpy(), tie.cpu().numpy()
            if every:
                check_f64(mar, cls, tie, ref, threads)
                assert h.last_recheck_count() == len(S)
            else:
                check_f32(mar, cls, ref, threads)
