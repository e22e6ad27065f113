"""Planes shared by activation prefix: layer widths around the tile sizes (16-row blocks, 32 rows a wave, 128 rows
a block, 64 inputs at a time, 256 inputs a list pass), one hidden layer (no prefixes), many layers (table growth),
skips into odd widths.  The FP64 records equal the oracle's bit for bit, whatever tile a prefix falls into."""
import numpy as np
import pytest

import oracle
from analyticmesh_amd import configs
from analyticmesh_amd.engine import march

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nodes", [
    [3, 24, 1], [3, 17, 16, 15, 1], [3, 33, 31, 32, 1], [3, 64, 63, 65, 1], [3, 129, 127, 1], [3, 30, 128, 130, 1],
    [3, 255, 40, 1], [3, 257, 40, 1], [3, 40, 260, 24, 1], [3, 24, 24, 24, 24, 24, 24, 24, 24, 1]])
@pytest.mark.parametrize("seeds", [1, 40])
def test_prefix_planes_bitexact(nodes, seeds):
    spec = configs.geometric(nodes, 0.5, 0.03, 5)
    pts = configs.seeds_fibonacci(spec, seeds)
    st = configs.mask_of(spec, pts)
    ref = oracle.run_oracle(spec, pts, st, precision="fp64", traversal="bfs", max_regions=12000)
    got = march(spec, pts, st, precision="fp64", max_regions=12000)
    n = min(len(got.masks), len(ref.masks))
    assert n > 50
    for k in ("masks", "tabs", "vpairs"):
        assert np.array_equal(getattr(got, k)[:n], getattr(ref, k)[:n]), k
    assert np.array_equal(got.info[:n, :6], ref.info[:n, :6])
    assert np.array_equal(got.verts[:n].view(np.uint64), ref.verts[:n].view(np.uint64))
