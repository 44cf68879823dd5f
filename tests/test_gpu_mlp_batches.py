"""The network's batched gradient kernel (MlpGradKernel) at the edges of its
16-sample tiles and of its 512 workgroups, against the FP64 oracle, and
training that does not depend on the order of its workgroups.

Bound: a gradient is a sum of n products of FP32 activations; each product
carries a few roundings of 2^-24 and its 64-long inner sums at most 64 of them,
so 1e-5 of the gradient's norm covers sums whose terms cancel by a factor of a
few."""
from __future__ import annotations

import sys
from pathlib import Path

import numpy as np
import pytest

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "oracle"))
import mlp_oracle as M  # noqa: E402

import finitevolumesolver_amd as fvs  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("huber", [0.0, 0.25])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 1000, 8192, 8209])
def test_gradients_at_tile_edges(cuda, n, huber):
    import torch
    net = fvs.LearnedNewtonGuess(seed=11)
    rng = np.random.default_rng(n)
    x = rng.uniform(-1.0, 1.0, (6, n)).astype(np.float32)
    t = rng.uniform(-1.0, 1.0, n).astype(np.float32)
    flag = (rng.random(n) < 0.2).astype(np.int32) if n > 1 else np.zeros(1, np.int32)
    g, loss = net.gradients(torch.from_numpy(x).to(cuda), torch.from_numpy(t).to(cuda),
                            torch.from_numpy(flag).to(cuda), huber)
    ref_loss, ref = M.loss_and_grad(net.get_params(), x, t, flag, huber)
    assert abs(loss - ref_loss) <= 1e-5 * abs(ref_loss)
    assert np.linalg.norm(g - ref) <= 1e-5 * np.linalg.norm(ref)


def test_training_is_deterministic(cuda):
    runs = []
    for _ in range(2):
        net = fvs.LearnedNewtonGuess(seed=4)
        net.generate(20000, seed=9)
        hist = net.train(epochs=3, batch=1000, seed=5)
        runs.append((net.get_params(), hist))
    assert np.array_equal(runs[0][0], runs[1][0]) and np.array_equal(runs[0][1], runs[1][1])
    assert runs[0][1][-1] < runs[0][1][0]


def test_padding_columns_of_w1_are_ignored(cuda):
    """fvs_mlp_set_params takes any floats in the two padding columns of W1
    (inputs 6 and 7 do not exist): forward, inference, gradients and training
    are those of zero padding, and the columns are returned as they were set."""
    import torch
    rng = np.random.default_rng(3)
    n = 200
    x = torch.from_numpy(rng.uniform(-1.0, 1.0, (6, n)).astype(np.float32)).to(cuda)
    t = torch.from_numpy(rng.uniform(-1.0, 1.0, n).astype(np.float32)).to(cuda)
    flag = torch.zeros(n, dtype=torch.int32, device=cuda)
    prim = torch.from_numpy(np.stack([rng.uniform(0.5, 2.0, n), rng.uniform(-1, 1, n), 0.1 * rng.random(n),
                                      rng.uniform(5.0, 9.0, n), rng.uniform(0.5, 2.0, n),
                                      rng.uniform(0.8, 1.2, n)])).to(cuda)
    runs = []
    for pad in ((0.0, 0.0), (0.75, -2.0), (np.inf, np.nan)):
        net = fvs.LearnedNewtonGuess(seed=6)
        p = net.get_params()
        p[:512].reshape(64, 8)[:, 6:] = pad
        net.set_params(p)
        net.generate(4096, seed=2)
        out = [net.forward(x).cpu().numpy(), net.infer_pairs(2, 0, prim, prim.flip(1))[0].cpu().numpy(),
               *net.gradients(x, t, flag, 0.25), net.train(epochs=2, batch=512)]
        w = net.get_params()
        assert np.array_equal(w[:512].reshape(64, 8)[:, 6:], p[:512].reshape(64, 8)[:, 6:], equal_nan=True)
        runs.append(out + [fvs.newton_guess.unpack_params(w)["W1"], w[512:]])
    for other in runs[1:]:
        for a, b in zip(runs[0], other):
            assert np.all(np.isfinite(a)) and np.array_equal(a, b)
