"""Training kernels of the learned front-end where their tiles and splits
end: one 32-row tile, row counts that the splits of the weight gradients do
not divide, both class paddings (4 and 16), input widths around a tile of the
weight-gradient product, and hidden widths that run layer by layer.

Gradients against the float64 oracle with the tolerance of test_gpu_mlp.py
(2e-2 relative Frobenius norm per tensor, the BF16 roundings both sides
make); the same call twice must agree bit for bit (every sum has a fixed
order).
"""
import numpy as np
import pytest

from oracle import mlp_oracle as MO
from tensorqec.learned import HipMLP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_in,n_out,hidden,B", [
    (48, 4, 512, 32), (8, 1, 512, 64), (48, 4, 512, 1056), (130, 5, 512, 288), (512, 16, 512, 96),
    (80, 2, 512, 2080), (48, 4, 128, 160), (200, 16, 256, 1056),
])
def test_gradients_at_tile_edges(n_in, n_out, hidden, B):
    torch = pytest.importorskip("torch")
    rng = np.random.default_rng(B + n_in)
    mlp = HipMLP(n_in, n_out, hidden=hidden, seed=1)
    mlp.set_params(mlp.get_params() + rng.normal(0, 0.01, size=mlp.nparams).astype(np.float32))
    S = (rng.random((B, n_in)) < 0.2).astype(np.uint8)
    Q = rng.dirichlet(np.ones(n_out), size=B).astype(np.float32)
    dS, dQ = torch.from_numpy(S).to("cuda:0"), torch.from_numpy(Q).to("cuda:0")
    dG = torch.full((2, mlp.nparams + 1), float("nan"), dtype=torch.float32, device="cuda:0")
    # the second gradient starts at an odd address of the array
    loss = [mlp.gradients(dS.data_ptr(), dQ.data_ptr(), B, dG[i, :].data_ptr()) for i in (0, 1)]
    got = dG.cpu().numpy()
    assert loss[0] == loss[1]
    assert np.array_equal(got[0, :-1], got[1, :-1]) and np.isnan(got[:, -1]).all()
    X = np.zeros((B, mlp.kin))
    X[:, :n_in] = S
    ref_loss, _, ref = MO.forward_backward(mlp.unflatten(mlp.get_params()), X, Q)
    assert abs(loss[0] - ref_loss) < 1e-3 * max(1.0, abs(ref_loss))
    g = mlp.unflatten(got[0, :-1])
    for k, r in ref.items():
        # a single class has no gradient at all
        err = np.linalg.norm(g[k] - r) / np.linalg.norm(r) if n_out > 1 else np.linalg.norm(g[k])
        assert err < 2e-2, (k, err)
    assert not np.any(g["W1"][n_in:, :])
