"""Networks whose planes meet in common lines and points (weights on a coarse grid), and the same networks scaled
by powers of two: every plane is scaled exactly, so the march is the unscaled one.  The near walk's FP32 margin
must leave the ties to the scan's own expressions at every scale.  Records bit for bit against the oracle's."""
import numpy as np
import pytest

import oracle
from analyticmesh_amd import configs
from analyticmesh_amd.engine import march

pytestmark = pytest.mark.gpu


def _grid_net(nodes, seed, k):
    """Weights and biases small integers over 8 or 4; layer 1 and every bias times 2^k."""
    rng = np.random.default_rng(seed)
    W, B = [], []
    for l in range(len(nodes) - 1):
        lo, hi, den = (-3, 4, 1) if l == 0 else (-2, 3, 8)
        w = rng.integers(lo, hi, (nodes[l + 1], nodes[l])) / den
        if l == 0:
            w[np.abs(w).sum(1) == 0] = 1
        W.append(w * 2.0 ** k if l == 0 else w)
        B.append(rng.integers(-6, 7, nodes[l + 1]) / 4 * 2.0 ** k)
    return configs.NetSpec(nodes, W, B, f"grid {nodes} {seed} 2^{k}")


def _seed(nodes, seed):
    """A point of f = 0 by bisection between two random points, on the unscaled network."""
    spec, rng = _grid_net(nodes, seed, 0), np.random.default_rng(1000 + seed)
    f = lambda x: float(np.ravel(configs.forward_fp64(spec, x)[0])[0])
    while True:
        a, b = rng.normal(size=3), rng.normal(size=3)
        if f(a) < 0 < f(b):
            for _ in range(100):
                m = 0.5 * (a + b)
                a, b = (m, b) if f(m) < 0 else (a, m)
            return (0.5 * (a + b))[None]


@pytest.mark.parametrize("k", [0, -26, -30, -36, -42, -48, 20])
@pytest.mark.parametrize("nodes,seed", [([3, 143, 34, 1], 1), ([3, 230, 12, 1], 3), ([3, 265, 40, 1], 7),
                                        ([3, 48, 19, 10, 1], 8), ([3, 320, 64, 1], 2)])
def test_scaled_degenerate_networks(nodes, seed, k):
    pts = _seed(nodes, seed)
    spec = _grid_net(nodes, seed, k)
    st = configs.mask_of(spec, pts)
    ref = oracle.run_oracle(spec, pts, st, precision="fp64", traversal="bfs", max_regions=2000)
    got = march(spec, pts, st, precision="fp64", max_regions=2000)
    assert len(got.masks) == len(ref.masks) > 500
    for f in ("masks", "tabs", "vpairs"):
        assert np.array_equal(getattr(got, f), getattr(ref, f)), f
    assert np.array_equal(got.verts.view(np.uint64), ref.verts.view(np.uint64))
