"""One training step from the sample store, whose minibatch is the whole
store, so that the order of the shuffle matters for the summation only: the
loss is the oracle's, and the parameters move as Adam's first step does with
the gradient of the same rows given as features.

Adam's first step is -lr g / (|g| + 1e-8) for every parameter, so where the
sign of g is certain it is known. The two gradients have the same rounding
points; they differ by the order of fp32 sums and by features that round to the
other bf16 neighbour where the device's sine and the host's differ by an ulp
(one in about 2^15, by 2^-8): less than 1e-3 of a block's L2 norm, so the sign
is certain above twice that. The loss: 1e-3, as for given features."""
import numpy as np
import pytest

import qubatron_amd as q
from oracle import pyoracle as po
from tests import helpers as H
from tests.test_gpu_surrogate import BLOCKS
from tests.test_mlp_oracle import OFF, rand_params

pytestmark = pytest.mark.gpu
LR = 1e-3


@pytest.fixture(scope="module")
def scene():
    sc, pnt, nrm, col, nodes = H.scene(1, npoints=100000)
    ctx = q.Context(0)
    ctx.upload_octree(nodes)
    ctx.upload_model(col, nrm)
    ctx.upload_octree(np.zeros((1, 12), np.int32), dynamic=True)
    pos, ang = sc.poses(6, seed=5)
    lights = np.concatenate([np.asarray(sc.lights, np.float32).reshape(-1, 3)[:1], [[300.0, 1500.0, 1200.0]]])
    yield ctx, sc, [q.view(pos[i], ang[i], 160, 120, sc.basecube, sc.depth) for i in range(6)], lights.astype(np.float32)
    ctx.close()


@pytest.mark.parametrize("n", [16, 64, 80, 4096, 16400])  # less than a chunk of 64, one, one and a part, blocks of one, of two
def test_step_from_the_store(scene, n):
    ctx, sc, views, lights = scene
    p = rand_params(500 + n)
    ctx.surrogate_reserve(n, 1)
    for v in views * 3:  # about 9000 queries a round of the views
        ctx.render(v, lights, q.OUT_FLAGS | q.RENDER_COLLECT)
    assert ctx.surrogate_samples()[0] == n
    smp = ctx.surrogate_read_samples()
    x, y = po.mlp_features(smp[:, 0:3], smp[:, 3:6], smp[:, 6:9], sc.basecube), np.ascontiguousarray(smp[:, 9])
    print(f"[case] store of {n}, {int(y.sum())} lit", flush=True)
    ctx.surrogate_set_params(p)
    _, g = ctx.surrogate_grad(x, y)
    lo, go = po.mlp_backward(p, x, y, bf16=True)
    ctx.surrogate_set_params(p)
    loss = ctx.surrogate_train(sc.basecube, 1, n, LR, 9)
    assert abs(loss - lo) < 1e-3 * max(1.0, lo)
    d = ctx.surrogate_params().astype(np.float64) - p
    assert np.abs(d).max() <= LR * (1 + 1e-4) + 1e-7
    checked = 0
    for a, b in BLOCKS:
        s = slice(OFF[a], OFF[b])
        assert np.linalg.norm(g[s] - go[s]) <= 3e-2 * np.linalg.norm(go[s]) + 1e-7, a
        k = np.abs(g[s]) > max(2e-3 * float(np.linalg.norm(g[s])), 2e-6)  # |g| >= 1e-6 in both: the step is lr within 1 %
        np.testing.assert_allclose(d[s][k], -LR * np.sign(g[s][k]), rtol=0, atol=LR * 1e-2 + 1e-7, err_msg=a)
        checked += int(k.sum())
    assert checked > p.size // 4
