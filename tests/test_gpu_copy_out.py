"""Records and meshes copied into pinned and device arrays equal those copied into ordinary ones, through the
C-ABI: the networks of a batch in turn (their records are gathered on the context's stream right before the
copy, into a buffer that the previous network's still fill), then one context's records and mesh."""
import ctypes
import os

import numpy as np
import pytest

from analyticmesh_amd import configs
from analyticmesh_amd.engine import BatchEngine, march

pytestmark = pytest.mark.gpu

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "analyticmesh_amd", "libam.so")
VM = 20


def _lib():
    lib = ctypes.CDLL(LIB)
    P, I, LL = ctypes.c_void_p, ctypes.c_int, ctypes.POINTER(ctypes.c_longlong)
    lib.am_batch_create.argtypes = [P, I, P, P, I]
    lib.am_batch_run.argtypes = [P, P, P, I, P, P, P, ctypes.c_double, I, P]
    lib.am_batch_get_regions.argtypes = [P, I, LL] + [P] * 6
    lib.am_batch_destroy.argtypes = [P]
    lib.am_get_regions.argtypes = [P] * 7
    lib.am_combine.argtypes = [P, ctypes.c_double, P]
    lib.am_get_counts.argtypes = [P, LL, LL, LL, LL]
    lib.am_get_mesh.argtypes = [P] * 4
    return lib


def _arrays(shapes, where):
    import torch
    out = []
    for shape, dt in shapes:
        if where == "pinned":
            out.append(torch.empty(shape, dtype=dt, pin_memory=True).fill_(-1))
        else:
            out.append(torch.full(shape, -1, dtype=dt, device="cuda"))
    return out


def _record_shapes(n, words):
    import torch
    i, d = torch.int32, torch.float64
    return [((n, words), i), ((n, 8), i), ((n, VM + 1), i), ((n, VM, 3), d), ((n, VM, 2), i), ((n, 3), d)]


def _equal(got, want, tag):
    for k, (a, b) in enumerate(zip(got, want)):
        a = a.cpu().numpy()
        assert np.array_equal(a.view(np.uint8), np.ascontiguousarray(b).view(np.uint8)), f"{tag}: array {k}"


@pytest.mark.parametrize("where", ["pinned", "device"])
def test_batch_records(where):
    lib = _lib()
    specs = [configs.geometric(n, 0.5, 0.03, 3 + i) for i, n in enumerate([[3, 64, 48, 1], [3, 50, 40, 1], [3, 64, 64, 1]])]
    seeds = []
    for s in specs:
        p = configs.seeds_fibonacci(s, 8)
        seeds.append((p, configs.mask_of(s, p)))
    print(f"[copy out] batch {where}", flush=True)
    want = BatchEngine(specs, precision="fp64", vm=VM).run(seeds)
    keep, W, B = [], [], []

    def ptrs(arrays):
        return (ctypes.c_void_p * len(arrays))(*[a.ctypes.data for a in arrays])

    for s in specs:
        W += [np.ascontiguousarray(w, np.float64) for w in s.weights]
        B += [np.ascontiguousarray(b, np.float64) for b in s.biases]
    nodes = [np.array(s.nodes, np.int32) for s in specs]
    nn = np.array([len(n) for n in nodes], np.int32)
    pts = [np.ascontiguousarray(p, np.float64) for p, _ in seeds]
    sts = [np.ascontiguousarray(m, np.uint8) for _, m in seeds]
    ns = np.array([len(p) for p in pts], np.int32)
    h = ctypes.c_void_p()
    assert lib.am_batch_create(ctypes.byref(h), len(specs), nn.ctypes.data, ptrs(nodes), 2) == 0
    try:
        assert lib.am_batch_run(h, ptrs(W), ptrs(B), 1, ptrs(pts), ptrs(sts), ns.ctypes.data, 0.0, 0, None) == 0
        for turn in range(2):
            for i, s in enumerate(specs):
                ref = want.regions(i)
                got = _arrays(_record_shapes(len(ref["masks"]), s.W), where)
                n = ctypes.c_longlong()
                assert lib.am_batch_get_regions(h, i, ctypes.byref(n), *[a.data_ptr() for a in got]) == 0
                assert n.value == len(ref["masks"]) > 500
                _equal(got, [ref[k] for k in ("masks", "info", "tabs", "verts", "vpairs", "points")], f"net {i} turn {turn}")
    finally:
        lib.am_batch_destroy(h)


@pytest.mark.parametrize("where", ["pinned", "device"])
def test_context_records_and_mesh(where):
    import torch
    lib = _lib()
    spec = configs.geometric([3, 64, 48, 1], 0.5, 0.03, 3)
    p = configs.seeds_fibonacci(spec, 4)
    print(f"[copy out] context {where}", flush=True)
    r = march(spec, p, configs.mask_of(spec, p), precision="fp64", vm=VM)
    ctx = ctypes.c_void_p(r.engine._eng.ctx_address())
    got = _arrays(_record_shapes(len(r.masks), spec.W), where)
    assert lib.am_get_regions(ctx, *[a.data_ptr() for a in got]) == 0
    _equal(got, [r.masks, r.info, r.tabs, r.verts, r.vpairs, r.points], "records")
    V, F = r.combine()
    got = _arrays([(V.shape, torch.float64), (F.offsets.shape, torch.int32), (F.indices.shape, torch.int32)], where)
    assert lib.am_get_mesh(ctx, *[a.data_ptr() for a in got]) == 0
    _equal(got, [V, F.offsets, F.indices], "mesh")
