"""The training kernels (one tile kernel and its reduction) against the FP64
oracle at the edges of their 32-sample tiles and of one tile per compute
unit, and Adam training repeating itself bit for bit."""
import numpy as np
import pytest
import torch

from mt_amd import params as P
from mt_amd.engine import Engine, MLP_IN, MLP_OUT, MODE_STREAMED
from oracle import mlp_oracle as M
from tests.helpers import c1_batch

pytestmark = pytest.mark.gpu


def _samples(n, seed):
    rng = np.random.default_rng(seed)
    x = rng.uniform(-1.0, 1.0, (n, MLP_IN)).astype(np.float32)
    x[rng.random(n) < 0.5, 24:] = 0.0           # dilute beads: one block of eight neighbours
    return x, rng.normal(0.3, 0.5, (n, MLP_OUT)).astype(np.float32)


@pytest.mark.parametrize("n", [1, 16, 31, 32, 33, 777, 8192, 8225, 20001])
def test_loss_and_gradient_at_tile_edges(n):
    print(f"case MLP gradient n={n}", flush=True)
    x, t = _samples(n, n)
    w = M.init_weights(3) + np.random.default_rng(1).normal(0, 0.02, M.init_weights(3).shape).astype(np.float32)
    eng = Engine(P.derive(dict(P.TEA)), c1_batch(), mode=MODE_STREAMED)
    eng.mlp_set_weights(w)
    loss, g = eng.mlp_loss_grad(x, t)
    lo, go = M.loss_and_grad(w.astype(np.float64), x, t)
    # FP32 sums of at most 128 products per neuron (relative rounding a few
    # 2^-24 of the operands' size) and of n samples: 1e-5 of the norm
    assert loss == pytest.approx(lo, rel=1e-5)
    assert np.linalg.norm(g - go) <= 1e-5 * np.linalg.norm(go)
    assert np.abs(g - go).max() <= 1e-4 * np.abs(go).max()
    eng.close()


def test_training_repeats_and_follows_adam():
    print("case MLP training repeats bit for bit", flush=True)
    x, t = _samples(700, 5)
    out = []
    for _ in range(2):
        eng = Engine(P.derive(dict(P.TEA)), c1_batch(), mode=MODE_STREAMED)
        eng.mlp_set_weights(M.init_weights(3))
        losses = eng.mlp_train(x, t, iters=5, batch=300, lr=1e-3)
        out.append((losses, eng.mlp_get_weights()))
        eng.close()
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])
    # Adam (Kingma & Ba 2015) in FP64 over the same slices: samples 0-299,
    # 300-599, then from the top again
    w = M.init_weights(3).astype(np.float64)
    m, v = np.zeros_like(w), np.zeros_like(w)
    for k, (loss, lo) in enumerate(zip(out[0][0], (0, 300, 0, 300, 0)), 1):
        l64, g = M.loss_and_grad(w, x[lo:lo + 300], t[lo:lo + 300])
        assert loss == pytest.approx(l64, rel=1e-5)
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        w = w - 1e-3 * (m / (1 - 0.9 ** k)) / (np.sqrt(v / (1 - 0.999 ** k)) + 1e-8)
    # each step moves a weight by at most ~lr; rounding can turn a step only
    # where the gradient is near zero
    assert np.abs(out[0][1] - w).max() < 2e-3 and np.linalg.norm(out[0][1] - w) < 1e-4 * np.linalg.norm(w)


def test_training_gives_back_the_memory_of_a_large_set():
    """A set of 168 MB and as many losses as fit no small buffer: after the
    call only what small calls keep too is held."""
    print("case MLP training memory", flush=True)
    eng = Engine(P.derive(dict(P.TEA)), c1_batch(), mode=MODE_STREAMED)
    eng.mlp_set_weights(M.init_weights(3))
    x, t = np.zeros((400000, MLP_IN), np.float32), np.zeros((400000, MLP_OUT), np.float32)
    eng.mlp_train(x[:65536], t[:65536], iters=2, batch=500, lr=1e-3)
    before = torch.cuda.mem_get_info()[0]
    for _ in range(2):
        losses = eng.mlp_train(x, t, iters=3, batch=500, lr=1e-3)
        assert np.isfinite(losses).all() and len(losses) == 3
        assert before - torch.cuda.mem_get_info()[0] < 30e6
    # and small calls go on
    assert np.isfinite(eng.mlp_train(x[:1000], t[:1000], iters=2, batch=500, lr=1e-3)).all()
    assert eng.mlp_forward(x[:100]).shape == (100, MLP_OUT)
    eng.close()
