"""The register-resident kernels where their loads and their re-check end:
syndrome rows whose width allows 16-, 8-, 4- and 1-byte loads, at even and odd
addresses, single rows and ragged tiles, and batches in which every row is
re-checked in FP64 (more rows than a workgroup's waves take at a time).

FP32 marginals against the plan's FP64 kernel within the FP32 tolerance of
_parity.py; re-checked rows, and FP64 at an odd address against an aligned
call, bit for bit.
"""
import numpy as np
import pytest

from _parity import check_f32
from tensorqec import decoders as D
from tensorqec.codes import CSSTannerGraph, ShorCode, SteaneCode, SurfaceCode
from tensorqec.errors import css_syndrome_rows, iid_error, sample_depolarizing

pytestmark = pytest.mark.gpu

# syndrome bits: 6 (bytes), 8, 12 (words of 4), 14 (bytes), 24 (words of 8), 48 (words of 16)
CODES = [SteaneCode(), ShorCode(), SurfaceCode(3, 3), SurfaceCode(3, 5), SurfaceCode(5, 5), SurfaceCode(7, 7)]


def decode(torch, ct, S, mode, shift):
    n, w = S.shape
    buf = torch.zeros(n * w + 16, dtype=torch.uint8, device="cuda:0")
    buf[shift:shift + n * w] = torch.from_numpy(np.ascontiguousarray(S)).to("cuda:0").reshape(-1)
    mar = torch.full((n, 1 << ct.hip.n_out), -1.0, dtype=torch.float64, device="cuda:0")
    cls = torch.full((n,), -1, dtype=torch.int32, device="cuda:0")
    tie = torch.full((n,), 7, dtype=torch.uint8, device="cuda:0")
    ct.hip.decode_device(buf.data_ptr() + shift, n, mode, mar.data_ptr(), cls.data_ptr(), tie.data_ptr())
    return mar.cpu().numpy(), cls.cpu().numpy(), tie.cpu().numpy()


@pytest.mark.parametrize("code", CODES, ids=str)
@pytest.mark.parametrize("n", [1, 15, 65, 200])
def test_rows_widths_and_addresses(code, n):
    torch = pytest.importorskip("torch")
    t = CSSTannerGraph.from_code(code)
    em = iid_error(0.03, 0.02, 0.03, t.nq)
    ct = D.compile(D.TNMMAP(), t, em)
    S = css_syndrome_rows(sample_depolarizing(em, seed=31 + n, count=n), t)
    ref = decode(torch, ct, S, "spec_f64", 0)
    for shift in (0, 1, 4, 8):
        for a, b in zip(decode(torch, ct, S, "spec_f64", shift), ref):
            assert np.array_equal(a, b), shift
        mar, cls, _ = decode(torch, ct, S, "spec_f32", shift)
        check_f32(mar, cls, ref[0], f"{code} {shift}")
    assert ct.hip.spec_config()["reg"]
    # every row re-checked: the FP64 kernel's numbers
    ct.hip.set_tolerances(1e-12, 2.0)
    for threads in (64, 128, 256):
        ct.hip.set_spec(threads // 4, threads, False, 0, reg=True)
        for a, b in zip(decode(torch, ct, S, "spec_f32", 0), ref):
            assert np.array_equal(a, b), threads
        assert ct.hip.last_recheck_count() == n
