"""The gfx950 code that the library's kernels compile to (hipcc, no GPU)."""
import os
import re
import shutil
import subprocess

import pytest

from tensorqec import decoders as D
from tensorqec import lib as L
from tensorqec.codes import CSSTannerGraph, SteaneCode, SurfaceCode, ToricCode
from tensorqec.errors import iid_error

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "tensorqec.jl_amd", "csrc")


def assembly(source, tmp_path):
    hipcc = "/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else shutil.which("hipcc")
    if not hipcc:
        pytest.skip("hipcc not available")
    out = tmp_path / "kernels.asm"
    r = subprocess.run([hipcc, "-x", "hip", "--offload-arch=gfx950", "-O3", "-std=c++17", "--cuda-device-only", "-S",
                        str(source), "-o", str(out), "-I", os.path.join(REPO, "include"), "-I", CSRC, "-Xclang",
                        "-target-feature", "-Xclang", "-packed-fp32-ops"],
                       capture_output=True, text=True, timeout=600,
                       env={k: v for k, v in os.environ.items() if k != "LD_PRELOAD"})
    assert r.returncode == 0, r.stderr[-2000:]
    return out.read_text()


def vector_shifts(asm):
    """64-bit vector shifts whose amount is a vector register."""
    return re.findall(r"v_(?:lshl|lshr|ashr)rev_[bi]64\S*\s+v\[\d+:\d+\], v\d+, .*", asm)


@pytest.mark.parametrize("name", ["tqec_hip.hip", "sampler_hip.hip", "mlp_hip.hip"])
def test_library_kernels_shift_64_bits_by_no_vector_register(name, tmp_path):
    assert vector_shifts(assembly(os.path.join(CSRC, name), tmp_path)) == []


@pytest.mark.parametrize("kw", [dict(tile=64, threads=256, reg=True), dict(tile=64, threads=256, reg=True, fp64=True),
                                dict(tile=4, threads=64), dict(tile=1, threads=256, slab=True)], ids=str)
def test_generated_kernels_shift_64_bits_by_no_vector_register(kw, tmp_path):
    t = CSSTannerGraph.from_code(SurfaceCode(5, 5))
    src = D.compile(D.TNMMAP(), t, iid_error(0.02, 0.02, 0.02, t.nq)).hip.spec_source(tables_in_lds=False, **kw)
    f = tmp_path / "spec.hip"
    f.write_text("#include <hip/hip_runtime.h>\n" + src)
    assert vector_shifts(assembly(f, tmp_path)) == []


def test_layered_forward_waits_for_no_store_before_its_last(tmp_path):
    """Loads and stores share a counter, so a load waited for behind a store is
    a wait for the store: a hidden layer's epilogue loads nothing between the
    first of its stores and the last."""
    asm = assembly(os.path.join(CSRC, "mlp_hip.hip"), tmp_path)
    bodies = re.findall(r"^(\S*gemm_fwd_kernel\S*):(.*?)^\.Lfunc_end", asm, re.M | re.S)
    assert len(bodies) == 2                                # K steps of 64 and of 32
    for _, body in bodies:
        stores = body[body.index("global_store_short"):]
        assert stores.count("global_store_short") == 64 and "vmcnt" not in stores


@pytest.mark.parametrize("codes,wgs,scratch", [
    ((SteaneCode(), SurfaceCode(3, 3), SurfaceCode(5, 5)), 3, 0),
    ((SteaneCode(), SurfaceCode(3, 3), ToricCode(3, 3)), 3, 128),      # slab plan on MFMA
    ((SteaneCode(), SurfaceCode(3, 3), SurfaceCode(7, 7)), 2, 0),
], ids=["lds", "slab", "d7"])
def test_mixed_kernel_that_runs(codes, wgs, scratch, tmp_path):
    """256 threads, held to the workgroups per CU that its LDS allows (three at
    most), with no scratch but where three of a mix with a slab plan pay for it."""
    plans = []
    for c in codes:
        t = CSSTannerGraph.from_code(c)
        plans.append(D.compile(D.TNMMAP(), t, iid_error(0.02, 0.02, 0.02, t.nq)).hip)
    src = L.mixed_spec_source(plans)
    assert src == L.mixed_spec_source(plans, 256) and "__launch_bounds__(256, %d)" % wgs in src
    f = tmp_path / "mixed.hip"
    f.write_text("#include <hip/hip_runtime.h>\n" + src)
    asm = assembly(f, tmp_path)
    lds, used = (int(re.search(r"\.%s_segment_fixed_size: +(\d+)" % k, asm)[1]) for k in ("group", "private"))
    assert wgs * lds <= 160 * 1024 and (wgs == 3 or (wgs + 1) * lds > 160 * 1024) and used <= scratch
