"""Reduced forms whose vertices are all re-solved in FP64 march on the FP64 planes alone: the
records are the FP64 ray form's, and am_planes still gives the reduced planes (prepared on demand)."""
import numpy as np
import pytest

from _common import workload

pytestmark = pytest.mark.gpu


def _run(spec, pts, st, dtype, **kw):
    from analyticmesh_amd.engine import Engine
    cap = kw.pop("cap", None)
    eng = Engine(spec.nodes, **kw)
    if cap:
        eng.set_option("max_regions", cap)
    res = eng.run([np.ascontiguousarray(w, dtype) for w in spec.weights],
                  [np.ascontiguousarray(b, dtype) for b in spec.biases], pts.astype(dtype), st)
    return eng, res


@pytest.mark.parametrize("name,dtype,vm", [("sphere", np.float32, 20), ("sphere", np.float64, 8),
                                           ("deep", np.float32, 20)])
@pytest.mark.parametrize("form", [dict(precision="bf16x3"), dict(precision="fp32", reduced_vertices="fp64"),
                                  dict(precision="bf16x3", graph_levels=True)])
def test_resolved_forms_give_the_fp64_records(name, dtype, vm, form):
    spec, pts, st = workload(name, n_seeds=8)
    cap = 6000 if name == "deep" else None
    print(f"[resolved] {name} {np.dtype(dtype).name} vm {vm} {form}", flush=True)
    _, ref = _run(spec, pts, st, dtype, precision="fp64ray", vm=vm, cap=cap)
    eng, res = _run(spec, pts, st, dtype, vm=vm, cap=cap, **form)
    for a, b in ((res.masks, ref.masks), (res.tabs, ref.tabs), (res.vpairs, ref.vpairs), (res.verts, ref.verts)):
        assert np.array_equal(a, b)
    assert int(res.stats[9]) == len(res.masks)
    if form["precision"] == "fp32":
        other, _ = _run(spec, pts, st, dtype, precision="fp32", cap=100)
        for a, b in zip(eng.planes(ref.masks[:200], with_sigma=True), other.planes(ref.masks[:200], with_sigma=True)):
            assert np.array_equal(a, b)
