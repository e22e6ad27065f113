"""The near walk (one wave per region on the constraints closest to it) around its edges: constraint counts
just under, at and over one per lane, extra planes, small vertex caps, and faces too long for the near set.
The FP64 form is held to the oracle bit for bit, the certified form to its topology and 1e-12."""
import numpy as np
import pytest

import oracle
from _common import assert_same_topology, max_vertex_error
from analyticmesh_amd import configs
from analyticmesh_amd.engine import march

pytestmark = pytest.mark.gpu

BOX_W = np.concatenate([np.eye(3), -np.eye(3)]) + 1e-8
BOX_B = np.array([-2.0, -0.2, -0.2, 0.1, -0.2, -0.2])


def _case(nodes, box):
    spec = configs.geometric(nodes, 0.5, 0.03, 11)
    pts = configs.bisect_seed(spec, (1.0, 0.05, 0.02))[None]
    extra = dict(extra_w=BOX_W, extra_b=BOX_B) if box else {}
    return spec, pts, configs.mask_of(spec, pts), extra


@pytest.mark.parametrize("nodes,box,vm", [
    ([3, 31, 32, 1], False, 20), ([3, 32, 32, 1], False, 20), ([3, 33, 32, 1], False, 20),
    ([3, 29, 29, 1], True, 20), ([3, 30, 29, 1], True, 20), ([3, 64, 65, 1], False, 20),
    ([3, 64, 64, 64, 65, 1], True, 20), ([3, 40, 41, 1], False, 5), ([3, 40, 41, 1], False, 64)])
def test_near_walk_against_the_oracle(nodes, box, vm):
    spec, pts, st, extra = _case(nodes, box)
    ref = oracle.run_oracle(spec, pts, st, precision="fp64", traversal="bfs", vm=vm, **extra)
    a = march(spec, pts, st, precision="fp64", vm=vm, **extra)
    assert np.array_equal(a.masks, ref.masks)
    assert np.array_equal(a.info[:, :6], ref.info[:, :6])
    for k in ("tabs", "vpairs"):
        assert np.array_equal(getattr(a, k), getattr(ref, k)), k
    assert np.array_equal(a.verts.view(np.uint64), ref.verts.view(np.uint64))
    if vm < 10:
        return   # truncated polygons: which edges are cut off depends on the walk's first edge
    b = march(spec, pts, st, precision="fp64ray", vm=vm, **extra).records()
    assert_same_topology(b, ref.records())
    assert max_vertex_error(b, ref.records()) < 1e-12
