"""One-syndrome tiles with GEMM-shaped steps on FP32 MFMA, long contractions
split over the threads, and a slab plan's smaller intermediates in LDS: every
thread count (it sets the waves that share blocks, the threads that share a
contraction and the LDS that intermediates may take), from LDS and from a
slab, against the CPU oracle within the FP32 tolerance of _parity.py.  A slab
without MFMA steps keeps the generic kernel's bits whatever lies in LDS.
"""
import numpy as np
import pytest

from _parity import check_f32
from oracle.cexec import OraclePlan
from tensorqec import decoders as D
from tensorqec.circuits import detector_error_model_from_stim, rotated_memory_z
from tensorqec.codes import CSSTannerGraph, SurfaceCode, ToricCode
from tensorqec.errors import IndependentFlipError, css_syndrome_rows, iid_error, sample_depolarizing, sample_flips

pytestmark = pytest.mark.gpu

N = 67   # more than a workgroup's first tile, not a multiple of anything


def problem(name):
    if name == "dem":
        dem = detector_error_model_from_stim(rotated_memory_z(3, 3, 0.004))
        e = sample_flips(IndependentFlipError(dem.error_rates), 5, N)
        return D.compile(D.TNMMAP(optimizer=D.Dissection(seeds=1)), dem), (e @ dem.detector_matrix().T % 2).astype(np.uint8)
    t = CSSTannerGraph.from_code(ToricCode(3, 3) if name == "toric3" else SurfaceCode(5, 5))
    em = iid_error(0.02, 0.02, 0.02, t.nq)
    return D.compile(D.TNMMAP(), t, em), css_syndrome_rows(sample_depolarizing(em, seed=9, count=N), t)


def decode(torch, ct, S, mode="spec_f32"):
    dS = torch.from_numpy(np.ascontiguousarray(S)).to("cuda:0")
    mar = torch.full((len(S), 1 << ct.hip.n_out), -1.0, dtype=torch.float64, device="cuda:0")
    cls = torch.full((len(S),), -1, dtype=torch.int32, device="cuda:0")
    tie = torch.full((len(S),), 7, dtype=torch.uint8, device="cuda:0")
    ct.hip.decode_device(dS.data_ptr(), len(S), mode, mar.data_ptr(), cls.data_ptr(), tie.data_ptr())
    return mar.cpu().numpy(), cls.cpu().numpy(), tie.cpu().numpy()


@pytest.mark.parametrize("name", ["dem", "toric3"])
def test_gemm_tiles_vs_oracle(name):
    torch = pytest.importorskip("torch")
    ct, S = problem(name)
    ref, _, _ = OraclePlan(ct.plan).decode(S)
    mar, cls, _ = decode(torch, ct, S)
    check_f32(mar, cls, ref, name)
    cfg = ct.hip.spec_config()
    assert cfg["tile"] == 1 and cfg["mfma32"] and cfg["slab"] == (name == "toric3")
    for threads in (64, 128, 256):
        for slab in (False, True) if name == "dem" else (True,):
            ct.hip.set_spec(1, threads, False, 2, slab=slab, unroll=2, mfma32=True)
            mar, cls, _ = decode(torch, ct, S)
            check_f32(mar, cls, ref, f"{name} {threads} {slab}")


@pytest.mark.parametrize("tile,threads", [(1, 64), (2, 64), (4, 128), (16, 256)])
def test_slab_intermediates_in_lds_keep_the_bits(tile, threads):
    torch = pytest.importorskip("torch")
    ct, S = problem("surface5")
    ref = decode(torch, ct, S, "fused_f32")
    ct.hip.set_spec(tile, threads, False, 0, slab=True, unroll=2)
    for a, b in zip(decode(torch, ct, S), ref):
        assert np.array_equal(a, b)
