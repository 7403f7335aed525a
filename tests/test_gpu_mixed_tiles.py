"""The generated mixed-code kernel around its tile size and on both sides of
the tile count up to which one workgroup per CU takes the whole call: every
row bit-identical to the single-plan fused_f32 executor (the same arithmetic,
tiled otherwise)."""
import numpy as np
import pytest

from tensorqec import decoders as D
from tensorqec import lib as L
from tensorqec.codes import CSSTannerGraph, SteaneCode, SurfaceCode
from tensorqec.errors import css_syndrome_rows, iid_error, sample_depolarizing

pytestmark = pytest.mark.gpu


def test_tile_edges_and_counts():
    torch = pytest.importorskip("torch")
    plans = []
    for code, p in ((SteaneCode(), 0.05), (SurfaceCode(3, 3), 0.08), (SurfaceCode(5, 5), 0.08)):
        t = CSSTannerGraph.from_code(code)
        em = iid_error(p / 3, p / 3, p / 3, t.nq)
        plans.append((t, em, D.compile(D.TNMMAP(mode="fused_f32"), t, em)))
    mx = L.HipMixed([ct.hip for _, _, ct in plans], max_batches=16, max_rows=60000)
    mx.set_kernel(True)
    for sizes in ((1, 31, 32, 33, 63, 65), (16384, 1), (16385, 7, 20000, 3, 12000)):
        parts, table = [], []
        for k, n in enumerate(sizes):
            t, em, ct = plans[k % 3]
            S = css_syndrome_rows(sample_depolarizing(em, seed=3 + k, count=n), t)
            dS = torch.from_numpy(np.ascontiguousarray(S)).to("cuda:0")
            got = [torch.full((n, 4), -1.0, dtype=torch.float64, device="cuda:0"),
                   torch.full((n,), -1, dtype=torch.int32, device="cuda:0"),
                   torch.full((n,), 7, dtype=torch.uint8, device="cuda:0")]
            parts.append((ct, dS, n, got))
            table.append((k % 3, n, dS.data_ptr(), *(x.data_ptr() for x in got)))
        mx.decode_device(table)
        mx.last_call()
        for ct, dS, n, got in parts:
            ref = [torch.empty_like(x) for x in got]
            ct.hip.decode_device(dS.data_ptr(), n, "fused_f32", *(x.data_ptr() for x in ref))
            torch.cuda.synchronize()
            for a, b in zip(got, ref):
                assert torch.equal(a, b), n
