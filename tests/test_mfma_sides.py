"""GEMM-shaped steps on FP32 MFMA whichever operand holds the output's fastest
labels: a store's lanes lie along them (generated source), and the results of
every order, tile edge and block shape are the oracle's within the FP32
tolerance of _parity.py, from LDS and from a slab."""
import re

import numpy as np
import pytest

from _parity import check_f32
from oracle.cexec import OraclePlan
from tensorqec import lib as L
from tensorqec.planner import Plan


def product(ra, rb, rk, side, seed=1):
    """C[a, b] = sum_k A[a, k] B[k, b], A and B chosen by a syndrome bit each,
    then joined to a leaf chosen by a third bit over the labels of one side;
    the other side's are summed, and they are C's fastest."""
    rng = np.random.default_rng(seed)
    a, k, b = list(range(10, 10 + ra)), list(range(30, 30 + rk)), list(range(50, 50 + rb))
    o = [70, 71]
    rest = a if side else b
    leaves = [[0] + a + k, [1] + k + b, [2] + rest + o]
    data = [rng.uniform(0.1, 1.0, 1 << len(x)) for x in leaves]
    return Plan(3, leaves, data, [-1] * 3, [0, 3], [1, 2], [a + b, o], o, 3, {0: 0, 1: 1, 2: 2})


SHAPES = [(5, 5, 1), (6, 5, 4), (5, 7, 2), (7, 6, 5), (4, 4, 2), (4, 6, 3), (7, 4, 5)]


@pytest.mark.parametrize("side", [0, 1])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_lanes_lie_along_the_output(shape, side):
    h = L.HipPlan(product(*shape, side), tabulate_bits=0)
    src = h.spec_source(1, 128, False, slab=True, unroll=4, mfma32=True)
    step = next(s for s in src.split("{ // step ") if "__builtin_amdgcn_mfma_f32" in s)
    index = re.search(r"const unsigned c = tc \| (.*);", step)[1]
    rows = [int(x) for x in re.findall(r"\(\(\(i\) >> \d\) & 1u\) << (\d+)", index)]
    lanes = [int(x) for x in re.findall(r"\(unsigned\)\(l & \d+u\)\) >> \d\) & 1u\) << (\d+)", index)]
    assert len(lanes) == len(rows) == (5 if min(shape[:2]) >= 5 else 4)
    assert sum(x < 5 for x in rows) - sum(x < 5 for x in lanes) < 3


@pytest.mark.gpu
@pytest.mark.parametrize("side", [0, 1])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_orders_vs_oracle(shape, side):
    torch = pytest.importorskip("torch")
    plan = product(*shape, side)
    S = np.array([[(i >> j) & 1 for j in range(3)] for i in range(8)] * 9, np.uint8)
    ref, _, _ = OraclePlan(plan).decode(S)
    dS = torch.from_numpy(S).to("cuda:0")
    for threads in (64, 256):
        for slab in (False, True):
            h = L.HipPlan(plan, tabulate_bits=0)
            h.set_spec(1, threads, False, 2, slab=slab, unroll=4, mfma32=True)
            mar = torch.full((len(S), 4), -1.0, dtype=torch.float64, device="cuda:0")
            cls = torch.full((len(S),), -1, dtype=torch.int32, device="cuda:0")
            h.decode_device(dS.data_ptr(), len(S), "spec_f32", mar.data_ptr(), cls.data_ptr(), 0)
            check_f32(mar.cpu().numpy(), cls.cpu().numpy(), ref, f"{shape} {threads} {slab}")
