"""More seeds than one launch holds blocks of 64 threads for (2^26): the same seed over and over marches as one,
the last seeds count as much as the first."""
import numpy as np
import pytest

from analyticmesh_amd import configs
from analyticmesh_amd.engine import Engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1 << 20) + 3, (1 << 26) + 64])
def test_seeds_past_the_launch_limits(n):
    spec = configs.geometric([3, 6, 1], 0.5, 0.03, 1)
    two = np.stack([configs.bisect_seed(spec, (1.0, 0.0, 0.0)), configs.bisect_seed(spec, (-0.3, 1.0, 0.2))])
    states = configs.mask_of(spec, two).astype(np.uint8)
    two = two.astype(np.float32)
    w, b = ([np.asarray(a, np.float32) for a in arrays] for arrays in (spec.weights, spec.biases))
    want = Engine(spec.nodes, precision="fp64").run(w, b, two, states)
    # all but the last are the first seed: the visited set takes the first of the equal ones
    pts, st = np.repeat(two[:1], n, 0), np.repeat(states[:1], n, 0)
    pts[-1], st[-1] = two[1], states[1]
    print(f"[many seeds] {n}", flush=True)
    got = Engine(spec.nodes, precision="fp64").run(w, b, pts, st)
    for k in ("masks", "tabs", "vpairs", "verts", "points"):
        assert np.array_equal(getattr(got, k), getattr(want, k)), k
