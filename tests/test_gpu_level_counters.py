"""Levels launched ahead of their size give the records and the launch counts of levels launched when it is known
(graph_levels): also where a level has more than twice the regions of the one before and 256 more, so that what
was launched for it is not used, and at the end, where nothing is left for it."""
import numpy as np
import pytest

from analyticmesh_amd import configs
from analyticmesh_amd.engine import march

pytestmark = pytest.mark.gpu

LAUNCHES, LEVELS, CANDIDATES, CHAINS = 11, 6, 8, 31   # AM_STAT_*


@pytest.mark.parametrize("precision", ["fp64", "fp64ray", "fp32", "bf16x3"])
@pytest.mark.parametrize("n_seeds", [1, 200])
def test_counts_of_levels_launched_ahead(precision, n_seeds):
    spec = configs.geometric([3, 128, 128, 1], 0.5, 0.03, 7)
    pts = configs.seeds_fibonacci(spec, n_seeds)
    st = configs.mask_of(spec, pts)
    print(f"[level counters] {precision} {n_seeds} seeds", flush=True)
    known = march(spec, pts, st, precision=precision, graph_levels=True)
    if n_seeds > 1:
        first = len(march(spec, pts, st, precision=precision, max_regions=1).masks)
        both = len(march(spec, pts, st, precision=precision, max_regions=first + 1).masks)
        assert both - first > 2 * first + 256
    ahead = march(spec, pts, st, precision=precision)
    for k in ("masks", "tabs", "vpairs", "verts"):
        assert np.array_equal(getattr(ahead, k), getattr(known, k)), k
    for s in (LEVELS, CANDIDATES, LAUNCHES, CHAINS):
        assert ahead.stats[s] == known.stats[s], s
    assert ahead.stats[CHAINS] == ahead.stats[LEVELS]
