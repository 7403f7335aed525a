"""Host paths of the library over a stub of the HIP calls on host memory
(hip_stub.cpp): what they enqueue and wait for, and what they choose, without
a GPU."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)

PLAN = """
import sys
sys.path[:0] = [%r, %r]
import numpy as np
from tensorqec.learned import HipMLP
from tensorqec import decoders as D, lib as L
from tensorqec.codes import CSSTannerGraph, SurfaceCode
from tensorqec.errors import iid_error
t = CSSTannerGraph.from_code(SurfaceCode(3, 3))
ct = D.compile(D.TNMMAP(), t, iid_error(0.02, 0.02, 0.02, t.nq))
""" % (REPO, os.path.join(REPO, "tensorqec.jl_amd"))


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    hipcc = "/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else shutil.which("hipcc")
    if not hipcc:
        pytest.skip("hipcc not available")
    out = tmp_path_factory.mktemp("stub") / "libhip_stub.so"
    subprocess.run([hipcc, "-x", "hip", "--offload-arch=gfx950", "-O1", "-shared", "-fPIC", os.path.join(HERE, "hip_stub.cpp"), "-o", str(out)],
                   check=True, capture_output=True, timeout=300)
    return str(out)


def run(stub, code, **env):
    r = subprocess.run([sys.executable, "-c", PLAN + code], capture_output=True, text=True, timeout=300,
                       env={**os.environ, "LD_PRELOAD": " ".join([stub, os.environ.get("LD_PRELOAD", "")]).strip(),
                            **env})
    assert r.returncode == 0, r.stderr[-2000:]
    return r.stdout, [l[5:] for l in r.stderr.splitlines() if l.startswith("stub ")]


@pytest.mark.parametrize("rows", [3, 200000])          # pinned staging, copies of the caller's arrays
@pytest.mark.parametrize("fail", ["launch", "copy_out"])
@pytest.mark.parametrize("patterns", [False, True])
def test_failed_host_call_waits_for_its_copies(stub, rows, fail, patterns):
    """The staging buffer is written again by the next call, the caller's
    arrays may be gone: neither before the copies out of them have ended."""
    out, calls = run(stub, """
S = np.zeros((%d, ct.plan.n_syndrome_bits), np.uint8)
try:
    D.decode_batch(ct, S, error_patterns=%r)
except L.TqecError:
    print("failed")
""" % (rows, patterns), TQEC_STUB_FAIL=fail)
    assert out.strip() == "failed" and fail + " failed" in calls
    assert "wait" in calls[max(i for i, c in enumerate(calls) if c.startswith("copy_in")):]
    assert calls[-1] == "wait"


def test_mixed_kernel_does_not_depend_on_earlier_calls(stub):
    """A plan whose default FP32 tile runs GEMM-shaped steps on MFMA: asking
    for that default, or decoding with it, leaves the mixed-code kernel as it
    was; a pinned tile changes it."""
    out, _ = run(stub, """
from tensorqec.circuits import detector_error_model_from_stim, rotated_memory_z
hip = D.compile(D.TNMMAP(optimizer=D.Dissection(seeds=1)), detector_error_model_from_stim(rotated_memory_z(3, 3, 0.001))).hip
first = L.mixed_spec_source([ct.hip, hip], 256)
cfg = hip.spec_config()
print(cfg["mfma32"], cfg["slab"], L.mixed_spec_source([ct.hip, hip], 256) == first)
hip.set_spec(1, 256, False, mfma32=True)
print("mfma" in first, "mfma" in L.mixed_spec_source([ct.hip, hip], 256))
""")
    assert out.split() == ["True", "False", "True", "False", "True"]


@pytest.mark.parametrize("inference", [0, 1])
def test_training_runs_the_chosen_kernels(stub, inference):
    """Gradients and training steps run layer by layer where inference does."""
    _, calls = run(stub, """
S, Q, g = np.zeros((64, 8), np.uint8), np.full((64, 4), 0.25, np.float32), np.zeros(600000, np.float32)
m = HipMLP(8, 4, hidden=512, seed=1)
for k in (1 - %d, %d):
    m.set_inference(k)
    print("stub now", k, file=sys.stderr, flush=True)
    m.gradients(S.ctypes.data, Q.ctypes.data, 64, g.ctypes.data)
    m.train_step(S.ctypes.data, Q.ctypes.data, 64, 1e-3)
""" % (inference, inference))
    kernels = " ".join(c for c in calls[calls.index("now %d" % inference):] if c.startswith("kernel "))
    assert kernels.count("mlp_train_rows_kernel") == (2 if inference else 0)
    assert kernels.count("gemm_fwd_kernel") == (0 if inference else 6)
    assert kernels.count("mlp_dw_kernel") == 2


@pytest.mark.parametrize("occ,module,loads", [("2", 1, 1), ("12", 2, 2), ("11", 2, 2)])
def test_register_kernel_without_a_cap_that_the_compiler_missed(stub, occ, module, loads):
    """Held to two waves per SIMD (256 threads: two workgroups per CU): a build
    that does not reach them gives way to one without the cap."""
    _, calls = run(stub, """
cfg = ct.hip.spec_config()
assert cfg["reg"] and cfg["waves"] == 2 and cfg["threads"] == 256
D.decode_batch(ct, np.zeros((3, 8), np.uint8), mode="spec_f32")
assert ct.hip.spec_config() == cfg
""", TQEC_STUB_OCC=occ)
    assert calls.count("load") == loads and calls.count("unload") >= loads - 1
    assert [c for c in calls if c.startswith("module ")] == ["module %d" % module]


def test_tuning_keeps_a_default_that_nothing_beats(stub):
    run(stub, """
cfg, S = ct.hip.spec_config(), np.zeros((64, 8), np.uint8)
ct.hip.autotune("spec_f32", S.ctypes.data, 64)
assert ct.hip.spec_config() == cfg and cfg["reg"]
""")


def test_slab_intermediates_leave_lds_for_the_waves_asked_for(stub):
    """The LDS of a CU divided by the workgroups that `waves` waves per SIMD
    make, two at least."""
    _, calls = run(stub, """
from tensorqec.codes import ToricCode
t = CSSTannerGraph.from_code(ToricCode(4, 4))
hip = D.compile(D.TNMMAP(optimizer=D.TreeSA(ntrials=1, sweeps=50, restarts=1)), t, iid_error(0.02, 0.02, 0.02, t.nq)).hip
for waves in (2, 3, 4):
    hip.set_spec(1, 256, False, waves, slab=True, unroll=1)
    hip.decode(np.zeros((1, t.ns), np.uint8), "spec_f32")
""")
    lds = [int(c.split()[1]) for c in calls if c.startswith("lds ")]
    lds = [lds[0]] + lds[2:]                               # the second is the FP64 re-check's
    assert 53 * 1024 < lds[0] <= 80 * 1024 and 16 * 1024 < lds[1] <= 53 * 1024 and 16 * 1024 < lds[2] <= 40 * 1024


@pytest.mark.parametrize("k,mfma", [(1, False), (4, True)])
def test_default_tile_by_the_share_of_gemm_steps(stub, k, mfma):
    """A 32 x 32 product over k labels beside one of 2^13 entries without a
    contraction, too wide for registers: one-syndrome MFMA tiles only where the
    product is a quarter of the multiply-adds."""
    out, _ = run(stub, """
from tensorqec.planner import Plan
rng = np.random.default_rng(1)
a, b, k, x, o = range(10, 15), range(20, 25), range(30, 30 + %d), range(40, 53), [70]
leaves = [[0, *a, *k], [1, *k, *b], [2, *x], [3, *x], [0, *a[:2], *b[:2], *o], [1, *x[:3], *o]]
outs = [[*a, *b], [*x], [*o], [*o], [*o]]
p = Plan(6, leaves, [rng.uniform(0.1, 1, 1 << len(l)) for l in leaves], [-1] * 6, [0, 2, 6, 7, 8], [1, 3, 4, 5, 9],
         outs, [*o], 4, {i: i for i in range(4)})
cfg = L.HipPlan(p, tabulate_bits=0).spec_config()
print(cfg["reg"], cfg["mfma32"])
""" % k)
    assert out.split() == ["False", str(mfma)]


def test_partial_sums_push_no_plan_out_of_lds(stub):
    """A plan whose one-syndrome tile fills the LDS to the last 64 bytes, so
    that the partial sums of a split contraction have no room: it keeps an LDS
    tile, which calls without allocation and captured ones can take."""
    out, _ = run(stub, """
from tensorqec.planner import Plan
rng, lab, T = np.random.default_rng(1), 100, []
# pairs of tensors with `sh` labels in common, all made before the first pair is joined
for ra, rb, sh in ((15, 9, 9), (12, 11, 11), (10, 8, 8), (7, 4, 4)):
    a = list(range(lab, lab + ra))
    T += [a, a[:sh]]
    lab += ra
leaves, outs = [], [list(x) for x in T]
for i, x in enumerate(T):
    k, h = [lab, lab + 1], len(x) // 2
    lab += 2
    leaves += [[2 * i, *x[:h], *k], [2 * i + 1, *k, *x[h:]]]
n = len(leaves)
lhs, rhs = list(range(0, n, 2)), list(range(1, n, 2))
cur = []
for i in range(0, 8, 2):
    lhs, rhs = lhs + [n + i], rhs + [n + i + 1]
    outs.append([l for l in T[i] if l not in T[i + 1]])
    cur.append((n + 8 + i // 2, outs[-1]))
while len(cur) > 1:
    (x, a), (y, b) = cur[:2]
    lhs, rhs = lhs + [x], rhs + [y]
    outs.append(a + b)
    cur = [(n + len(outs) - 1, a + b)] + cur[2:]
p = Plan(n, leaves, [rng.uniform(0.1, 1, 1 << len(l)) for l in leaves], [-1] * n, lhs, rhs, outs, outs[-1], 16,
         {i: i for i in range(16)})
hip = L.HipPlan(p, tabulate_bits=0)
size = [hip.spec_source(1, 64, False, unroll=4, mfma32=m).split("smem[")[1].split("]")[0] for m in (False, True)]
assert int(size[0]) <= 160 * 1024 < int(size[1]), size
print(hip.spec_config()["slab"])
""")
    assert out.strip() == "False"
