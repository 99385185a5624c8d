"""Photon tree builds (GPU): box pyramid, hierarchy and wide collapse at primitive counts around
their group, block and subtree sizes, against the oracle's brute force."""
import numpy as np
import pytest

from gpuupbp_amd import renderer as gpu
from oracle import oracle_py

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 7, 8, 9, 63, 65, 127, 128, 129, 511, 512, 513, 4095, 4097, 33000, 300001])
@pytest.mark.parametrize("shape", ["uniform", "piled", "skewed"])
def test_build_sizes_match_brute_force(n, shape):
    rng = np.random.default_rng(n)
    p = rng.uniform(-1, 1, (n, 3))
    if shape == "piled":  # equal codes: the hierarchy splits them by index
        p[rng.uniform(size=n) < 0.7] = 0.25
    elif shape == "skewed":  # a deep tree: a chain of ever smaller clusters
        p = p * 2.0 ** -rng.integers(0, 28, (n, 1))
    pts = p.astype(np.float32)
    r = 0.3 if n < 100 else (0.05 if n < 5000 else 0.01)
    if shape == "skewed" and n >= 100:
        r = 1e-4  # not the whole pile: a walk that meets everything outgrows its stack
        p = p[np.abs(p).max(axis=1) > 2e-4]
    at = p[rng.integers(0, len(p), 40)] + rng.normal(size=(40, 3)) * 0.1 * r
    d = rng.normal(size=(40, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    q = np.hstack([at - 0.5 * d, d, np.zeros((40, 1)), np.ones((40, 1))]).astype(np.float32)
    oo, oi = oracle_py.range_query(1, pts, q, r)
    assert n < 3 or oo[-1] > 0
    for wide in (False, True):
        go, gi = gpu.range_query(1, pts, q, r, wide=wide)
        assert np.array_equal(go, oo), wide
        for i in range(40):
            assert np.array_equal(np.sort(gi[go[i]:go[i + 1]]), np.sort(oi[oo[i]:oo[i + 1]]))
