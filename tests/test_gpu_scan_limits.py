"""As many constraints as the FP64 candidate scan's LDS holds (its planes, sort keys and records within 160 KiB),
and one more: the largest counts march as the oracle does, past them am_run fails with AM_ERR_CAPACITY (4)."""
import numpy as np
import pytest

import oracle
from analyticmesh_amd import configs
from analyticmesh_amd.engine import march

pytestmark = pytest.mark.gpu

LDS = 160 * 1024


def _scan_lds(C, words, vm):
    a16 = lambda x: (x + 15) & ~15
    sort = 64
    while sort < C:
        sort *= 2
    head = a16(32 * C + 12 * sort + 4 * ((C + 31) // 32) + 4 * words)
    return head + a16(24 * vm) + a16(8 * vm) + a16(4 * (vm + 2))


def _case(nodes, C, seed):
    spec = configs.geometric(nodes, 0.5, 0.03, 11)
    pts = configs.bisect_seed(spec, (1.0, 0.05, 0.02))[None]
    rng = np.random.default_rng(seed)
    n = rng.normal(size=(C - spec.L, 3))
    n /= np.linalg.norm(n, axis=1)[:, None]
    return spec, pts, configs.mask_of(spec, pts), dict(extra_w=n, extra_b=-(n @ pts[0]) - rng.uniform(0.2, 0.6, len(n)))


@pytest.mark.parametrize("precision", ["fp64", "fp64ray"])
@pytest.mark.parametrize("nodes,vm", [([3, 16, 1], 64), ([3, 16, 1], 3), ([3, 30, 30, 1], 20)])
def test_largest_constraint_counts(nodes, vm, precision):
    words = (sum(nodes[1:-1]) + 31) // 32
    most = max(C for C in range(2049, 4097) if _scan_lds(C, words, vm) <= LDS)
    for C in (most - 1, most):
        spec, pts, st, extra = _case(nodes, C, C)
        print(f"[scan limits] {nodes} vm {vm} {precision} C {C}", flush=True)
        ref = oracle.run_oracle(spec, pts, st, precision="fp64", traversal="bfs", max_regions=100, vm=vm, **extra)
        got = march(spec, pts, st, precision=precision, max_regions=100, vm=vm, **extra)
        if precision == "fp64":
            assert len(got.masks) == len(ref.masks) > 3
            for k in ("masks", "tabs", "vpairs"):
                assert np.array_equal(getattr(got, k), getattr(ref, k)), k
            assert np.array_equal(got.verts.view(np.uint64), ref.verts.view(np.uint64))
        elif vm >= 20:
            assert got.records().visited() == ref.records().visited()
    spec, pts, st, extra = _case(nodes, most + 1, 0)
    with pytest.raises(RuntimeError, match="am error 4"):
        march(spec, pts, st, precision=precision, max_regions=100, vm=vm, **extra)
