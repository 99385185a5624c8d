"""Batch sizes at the edges of the network kernels' tiles (GPU): 16-row forward tiles, 32-row gradient
steps, 256-row and larger chunks per block."""
import numpy as np
import pytest

from gpuupbp_amd import renderer as gpu
from oracle import oracle_py
from test_gpu_mlp import _samples

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 31, 33, 255, 256, 257, 1000, 4097, 32769, 40000])
def test_gradient_and_forward_at_tile_edges(n):
    m = gpu.Mlp(seed=6)
    s = _samples(np.random.default_rng(n), n)
    loss, g = m.loss_grad(s)
    # the batch twice over: the deltas are exactly half (a power of two), each row lands in another
    # tile and chunk, and only the order of the FP32 sums changes
    loss2, g2 = m.loss_grad(np.tile(s, (2, 1)))
    assert abs(loss - loss2) <= 1e-5 * abs(loss) + 1e-6
    assert np.linalg.norm(g - g2) <= 1e-5 * np.linalg.norm(g)
    _, go = oracle_py.mlp_loss_grad(m.params().astype(np.float64), s)
    # BF16 operands: seven products (four forward, three backward) of operands rounded by 2^-9 each
    # are off by up to 7 * 2 * 2^-9 = 2.7% of the samples' own gradients, whose mean is shorter than
    # they are (by up to 8 here: the scattered directions are uniform), so 0.22 of it
    assert np.linalg.norm(g - go) <= 0.22 * np.linalg.norm(go)
    f = np.ascontiguousarray(s[:, :6])
    o = oracle_py.mlp_forward(m.params().astype(np.float64), f)
    got = m.forward(f)
    assert got.shape == (n, 40)
    assert np.linalg.norm(got - o) <= 0.03 * np.linalg.norm(o)
    m.close()
