"""The max-product kernel with a wave per syndromes against the generic
kernel (configurations and log-maxima equal: the same comparisons in the same
order), where it can go wrong: one row, ragged groups, more rows than run at
once, configurations cut short, no log-maxima, and calls repeated (a wave's
second group starts from what the first left behind)."""
import numpy as np
import pytest

from tensorqec.codes import CSSTannerGraph, ShorCode, SteaneCode, SurfaceCode
from tensorqec.errors import css_syndrome_rows, iid_error, sample_depolarizing
from tensorqec.tnmap import TNMAP, compile_tnmap

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("code", [SteaneCode(), ShorCode(), SurfaceCode(3, 3), SurfaceCode(3, 5), SurfaceCode(5, 5)], ids=str)
@pytest.mark.parametrize("fac", [True, False])
def test_wave_map_kernel(code, fac):
    torch = pytest.importorskip("torch")
    t = CSSTannerGraph.from_code(code)
    em = iid_error(0.02, 0.01, 0.03, t.nq)
    ct = compile_tnmap(TNMAP(factorize=fac), t, em)
    n = 40001
    S = css_syndrome_rows(sample_depolarizing(em, 9 + t.nq, n), t)
    dS = torch.from_numpy(np.ascontiguousarray(S)).to("cuda:0")

    def run(rows, nv, with_logp=True):
        cfg = torch.full((rows, nv), 9, dtype=torch.uint8, device="cuda:0")
        lp = torch.full((rows,), 7.0, dtype=torch.float64, device="cuda:0")
        ct.hip.map_decode_device(dS.data_ptr(), rows, nv, cfg.data_ptr(), lp.data_ptr() if with_logp else 0)
        return cfg.cpu().numpy(), lp.cpu().numpy()

    nv = ct.qubit_num
    ct.hip.set_map_kernel(False)
    ref = run(n, nv)
    ct.hip.set_map_kernel(True)
    for rows in (1, 2, 15, 17, 63, 1000, n, n, n):
        cfg, lp = run(rows, nv)
        assert np.array_equal(cfg, ref[0][:rows]) and np.array_equal(lp, ref[1][:rows]), rows
    assert ct.hip.map_kernel() == (True, "")
    cfg, lp = run(1000, nv - 3, with_logp=False)
    assert np.array_equal(cfg, ref[0][:1000, :nv - 3]) and np.all(lp == 7.0)
