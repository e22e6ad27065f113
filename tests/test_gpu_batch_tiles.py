"""A batch level's kernels at their edges: more networks than one block finds the regions of, layers just
at and over what four waves cover, and more constraints than the near walk takes whole.  Every network's
records are those of its own march (both run the canonical planes: bit for bit)."""
import numpy as np
import pytest

from analyticmesh_amd import configs
from analyticmesh_amd.engine import BatchEngine, march

pytestmark = pytest.mark.gpu

WIDTHS = {
    "70 small": [[3, 20 + i % 5, 18 + i % 4, 1] for i in range(70)],
    "128 and 129 wide": [[3, 16, 128, 9, 1], [3, 129, 17, 1], [3, 15, 16, 17, 1]],
    "256 and 257 constraints": [[3, 200, 56, 1], [3, 200, 57, 1], [3, 40, 1]],
    "256 constraints": [[3, 192, 64, 1], [3, 33, 31, 32, 1]],
}


@pytest.mark.parametrize("precision", ["fp64", "fp64ray"])
@pytest.mark.parametrize("name", list(WIDTHS))
def test_batch_records_equal_single_marches(name, precision):
    specs = [configs.geometric(n, 0.5, 0.04, 20 + i) for i, n in enumerate(WIDTHS[name])]
    seeds = []
    for s in specs:
        p = configs.seeds_fibonacci(s, 3)
        seeds.append((p, configs.mask_of(s, p)))
    print(f"[batch tiles] {name} {precision}", flush=True)
    res = BatchEngine(specs, precision=precision).run(seeds)
    for i, (s, (p, st)) in enumerate(zip(specs, seeds)):
        r, g = march(s, p, st, precision=precision), res.regions(i)
        for k in ("masks", "tabs", "vpairs", "verts"):
            np.testing.assert_array_equal(g[k], getattr(r, k), err_msg=f"net {i} {k}")
