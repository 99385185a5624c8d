"""Batch sizes at the edges of the network kernels' tiles (GPU): 16-row forward tiles, 32-row gradient
steps, 256-row and larger chunks per block."""
import numpy as np
import pytest

from gpuupbp_amd import renderer as gpu
from oracle import oracle_py
from test_gpu_mlp import _samples

pytestmark = pytest.mark.gpu


SHAPES = [(64, 51), (64, 64), (64, 64), (40, 64)]


def _bf16(x):
    """Rounded to BF16, to nearest even, as the kernels round FP32 values."""
    u = np.asarray(x, np.float32).view(np.uint32).astype(np.uint64)
    return ((u + 0x7fff + ((u >> 16) & 1)) >> 16 << 16).astype(np.uint32).view(np.float32).astype(np.float64)


def _rounded_gradient(params, s):
    """The gradient's slices (weights and biases of each layer) in 64 bits with the kernels' BF16
    roundings: weights, encoded inputs, activations and deltas."""
    at, ws, bs = 0, [], []
    for rows, cols in SHAPES:
        ws.append(_bf16(params[at:at + rows * cols]).reshape(rows, cols))
        at += rows * cols
        bs.append(params[at:at + rows].astype(np.float64))
        at += rows
    n = len(s)
    x = np.zeros((n, 51))
    for j in range(3):
        for k in range(8):
            a = (np.float32(1 << k) * np.float32(np.pi) * s[:, j]).astype(np.float64)  # FP32 product
            x[:, (j * 8 + k) * 2], x[:, (j * 8 + k) * 2 + 1] = np.sin(a), np.cos(a)
    x[:, 48:] = s[:, 3:6]
    acts = [_bf16(x)]
    for k in range(3):
        acts.append(_bf16(np.maximum(acts[-1] @ ws[k].T + bs[k], 0.0)))
    o = (acts[3] @ ws[3].T + bs[3]).reshape(n, 8, 5)
    w, weight = s[:, 6:9].astype(np.float64), s[:, 9].astype(np.float64)
    norm = np.linalg.norm(o[:, :, :3], axis=2)
    mu = o[:, :, :3] / norm[:, :, None]
    kap = np.logaddexp(0.0, o[:, :, 3]) + 0.01
    e = np.exp(o[:, :, 4] - o[:, :, 4].max(axis=1, keepdims=True))
    pi = e / e.sum(axis=1, keepdims=True)
    cd = np.einsum("nlk,nk->nl", mu, w)
    v = kap / (2 * np.pi * -np.expm1(-2 * kap)) * np.exp(kap * (cd - 1))
    gam = pi * v / (pi * v).sum(axis=1, keepdims=True)
    g = np.zeros((n, 8, 5))
    g[:, :, 4] = pi - gam
    g[:, :, 3] = -gam * (1 / kap - 2 / np.expm1(2 * kap) + cd - 1) / (1 + np.exp(-o[:, :, 3]))
    g[:, :, :3] = (w[:, None, :] - mu * cd[:, :, None]) * (-gam * kap / norm)[:, :, None]
    delta = _bf16((g * (weight / n)[:, None, None]).reshape(n, 40))
    out = []
    for k in (3, 2, 1, 0):
        out = [delta.T @ acts[k], delta.sum(axis=0)] + out
        if k:
            delta = _bf16((delta @ ws[k]) * (acts[k] > 0))
    return out


@pytest.mark.parametrize("n", [1, 16, 17, 31, 33, 255, 257, 1000, 4097, 32769])
def test_every_layers_gradient_matches_the_rounded_one(n):
    m = gpu.Mlp(seed=6)
    s = _samples(np.random.default_rng(n), n)
    _, g = m.loss_grad(s)
    at = 0
    for want in _rounded_gradient(m.params(), s):
        got = g[at:at + want.size].reshape(want.shape).astype(np.float64)
        at += want.size
        # The same operands, so only FP32 sums and functions differ (1e-6 to 1e-5 relative), and the
        # roundings they tip: a share of 1e-5 / 2^-8 of the values moves by 2^-8, 2e-4 of a norm; with a
        # single row, one such value may carry the norm: 2^-8.
        assert np.linalg.norm(got - want) <= (4e-3 if n < 64 else 1e-3) * np.linalg.norm(want), (n, want.shape)
    assert at == g.size
    m.close()


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
