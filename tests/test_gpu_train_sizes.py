"""The training kernels at the batch sizes where they can go wrong: less than
a fragment group, a chunk of 64 samples and one more, more chunks than blocks
(a block then keeps its gradients over several chunks). The gradient and loss
agree with the oracle's to the tolerance of the other gradient tests (MFMA
summation order at bf16 rounding points: 3e-2 in relative L2 norm per
parameter block, cosine > 0.999), and one Adam step from that gradient moves
the parameters, and so the next forward pass, as the oracle's."""
import numpy as np
import pytest

from oracle import pyoracle as po
from tests.test_gpu_surrogate import BLOCKS, _rand_features
from tests.test_mlp_oracle import OFF, rand_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 64, 65, 129, 16384, 16400])
def test_gradient_and_step_sizes(gpu_ctx, n):
    p = rand_params(300 + n)
    gpu_ctx.surrogate_set_params(p)
    _, _, _, x = _rand_features(301 + n, n)
    y = (np.random.default_rng(302 + n).uniform(size=n) < 0.4).astype(np.float32)
    print(f"[case] n={n}", flush=True)
    loss, g = gpu_ctx.surrogate_grad(x, y)
    lo, go = po.mlp_backward(p, x, y, bf16=True)
    assert abs(loss - lo) < 1e-3 * max(1.0, lo)
    for a, b in BLOCKS:
        s = slice(OFF[a], OFF[b])
        assert np.linalg.norm(g[s] - go[s]) <= 3e-2 * np.linalg.norm(go[s]) + 1e-7, a
    assert float(g @ go) > 0.999 * float(np.linalg.norm(g) * np.linalg.norm(go))
    gpu_ctx.surrogate_step(x, y, 1e-3)
    ref, m, v = p.copy(), np.zeros_like(p), np.zeros_like(p)
    po.mlp_adam(ref, g, m, v, 1, lr=1e-3)
    np.testing.assert_allclose(gpu_ctx.surrogate_params(), ref, rtol=0, atol=1e-6)
    k = min(n, 500)
    pg, (pr, _) = gpu_ctx.surrogate_forward(x[:k]), po.mlp_forward(ref, x[:k], bf16=True)
    assert np.median(np.abs(pg - pr)) < 1e-3 and np.abs(pg - pr).max() < 2e-2
