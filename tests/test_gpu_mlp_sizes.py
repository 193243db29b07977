"""The network's fused passes at the edges of their tiles (rows around the 32
of a workgroup and the 128 and 512 of the gradient chunks, widths that fill
64, 128 or 256 columns partly, inputs with unaligned rows, many outputs) and
the GEMM-per-layer form past 256 inputs, against the CPU oracle with the
bounds of test_gpu_mlp.py (outputs and gradients 2e-3 in relative L2: BF16
operands, sums in another order)."""
import os
import sys

import numpy as np
import pytest
import torch

from lsd.gpu import Mlp

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mlp_ref  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_in,width,n_out,rows", [
    (92, 256, 10, 1), (92, 256, 10, 33), (92, 256, 10, 513), (92, 250, 10, 129), (17, 48, 3, 640), (93, 200, 33, 127),
    (92, 128, 10, 1025), (256, 256, 256, 96), (92, 64, 64, 31), (1, 16, 1, 512), (300, 256, 10, 200), (92, 260, 10, 65),
    (300, 20, 3, 7), (300, 20, 3, 8), (92, 64, 65, 1025)])
def test_sizes(n_in, width, n_out, rows):
    rng = np.random.default_rng(rows + width)
    m = Mlp(n_in, width, n_out, seed=3)
    p = m.params()
    X = rng.standard_normal((rows, n_in)).astype(np.float32)
    T = rng.standard_normal((rows, n_out)).astype(np.float32)
    y = m.forward(X)
    yo, _ = mlp_ref.forward(p, X, n_in, width, n_out, rb=True)
    assert np.linalg.norm(y - yo) <= 2e-3 * np.linalg.norm(yo)
    loss, g = m.grad(X, T)
    lo, go = mlp_ref.loss_and_grad(p, X, T, n_in, width, n_out, rb=True)
    assert abs(loss - lo) <= 1e-3 * lo
    assert np.linalg.norm(g - go) <= 2e-3 * np.linalg.norm(go)
    # a step of training on a batch that leaves a short rest: the losses are
    # those of the batches
    batch = max(1, 2 * rows // 3)
    losses = m.train(X, T, batch, 2, 0.0)
    part = [m.grad(X[:batch], T[:batch])[0], m.grad(X[batch:], T[batch:])[0] if rows > batch else m.grad(X, T)[0]]
    assert np.array_equal(losses, np.array(part, dtype=np.float32))
    m.close()


@pytest.mark.parametrize("width", [1, 16, 63, 64, 100, 250])
def test_infinite_inputs(width):
    """A row with an infinite input gives what the layers' definition gives:
    with positive weights +inf, not the NaN of an infinity times the zeros
    that pad the width; the other rows keep their results."""
    m = Mlp(4, width, 3, seed=1)
    m.set_params(np.full(m.n_params, 0.125, dtype=np.float32))
    X = np.random.default_rng(2).standard_normal((40, 4)).astype(np.float32)
    want = m.forward(X)
    X[[5, 39], 2] = np.inf
    y = m.forward(X)
    assert np.all(y[[5, 39]] == np.inf)
    rest = np.ones(40, dtype=bool)
    rest[[5, 39]] = False
    assert np.array_equal(y[rest], want[rest])
    m.close()


def test_memory_and_losses_of_large_batches():
    """The loss partials add little to the activations (X, Y, T and dY, six
    arrays of the width; 100000 floats of partials a step here, for which 256
    steps would take 102 MB), and the losses are right when they are fetched
    every few steps: with no learning rate those of the two batches in turn."""
    m = Mlp(4, 4, 64, seed=5)
    rows = 400000
    rng = np.random.default_rng(6)
    X = rng.standard_normal((rows, 4)).astype(np.float32)
    T = rng.standard_normal((rows, 64)).astype(np.float32)
    m.forward(X[:8])
    free = torch.cuda.mem_get_info()[0]
    m.grad(X, T)
    used = free - torch.cuda.mem_get_info()[0]
    assert used <= 4 * rows * (4 + 3 * 64 + 6 * 4) + (32 << 20)
    half = [m.grad(X[:rows // 2], T[:rows // 2])[0], m.grad(X[rows // 2:], T[rows // 2:])[0]]
    m.close()
    m = Mlp(4, 4, 64, seed=5)
    losses = m.train(X, T, rows // 2, 45, 0.0)
    assert np.array_equal(losses, np.array((half * 23)[:45], dtype=np.float32))
    m.close()
