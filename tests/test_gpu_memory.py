"""Memory of ended engines: kept for the next one, given back by trim_memory() and by the drop-in Destroy(), not
counted as used when the planes' storage grows on a nearly full device; and marches whose planes' table starts
over again and again there give the same topology."""
import gc

import numpy as np
import pytest

from _common import workload
from analyticmesh_amd import configs
from analyticmesh_amd.engine import Engine, march, trim_memory

pytestmark = pytest.mark.gpu

MB = 1 << 20
RESTARTS = 39   # AM_STAT_PREFIX_RESTARTS


def _free():
    import torch
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def _base():
    """Free memory with nothing kept (after a first march, so that the kernels are loaded)."""
    march(*workload("polytope"))
    gc.collect()
    trim_memory()
    return _free()


def test_trim_gives_back_what_ended_engines_left():
    base = _base()
    spec, pts, st = workload("sphere")
    print("[memory] trim", flush=True)
    live = march(spec, pts, st)
    masks = live.masks.copy()
    with_live = _free()
    march(spec, pts, st, table_log2=28)      # a visited table of 1 GiB
    gc.collect()
    assert with_live - _free() > 900 * MB     # kept for the next engine
    trim_memory()
    assert with_live - _free() < 64 * MB
    # the live engine still has its records, and marches again
    assert np.array_equal(live._eng.regions(live.Wd)["masks"], masks)
    live.combine()
    again = march(spec, pts, st)
    assert np.array_equal(again.masks, masks)
    del live, again
    gc.collect()
    trim_memory()
    assert abs(base - _free()) < 64 * MB


def test_destroy_of_the_drop_in_frees():
    import torch
    from analyticmesh_amd import cuam
    spec = configs.deep(0)
    pts = configs.bisect_seed(spec, (1.0, 0.0, 0.0))[None]
    t = lambda a: torch.tensor(np.asarray(a), dtype=torch.float64, device="cuda")
    W, B, p, none = [t(w) for w in spec.weights], [t(b) for b in spec.biases], t(pts), t(np.zeros((0, 3)))
    states = torch.tensor(configs.mask_of(spec, pts), device="cuda").bool()
    _base()

    def use():
        print("[memory] drop-in", flush=True)
        cuam.Init("float64", spec.nodes, torch.zeros((len(spec.nodes) - 2, 1), dtype=torch.int32), 0)
        cuam._S["engine"].set_option("max_regions", 30000)
        cuam.AnalyticMarching(W, B, states, p, [], none, none[:, 0].contiguous(), 0.0, False)
        used = _free()
        cuam.Destroy()
        gc.collect()
        return used, _free()

    first, second = use(), use()      # (the first loads kernels)
    assert first[1] - second[0] > 256 * MB
    assert first[1] - second[1] < 16 * MB


def test_planes_storage_on_a_nearly_full_device():
    """The 4x256 network's planes take more than their storage holds.  With 2 GiB over the quarter that stays
    free, and as much kept of ended engines, it is as large as with nothing kept; the marches agree."""
    import torch
    base = _base()
    spec, pts, st = workload("deep")
    args = ([np.asarray(w, np.float64) for w in spec.weights], [np.asarray(b, np.float64) for b in spec.biases], pts, st)

    def run():
        r = Engine(spec.nodes, precision="fp64ray").run(*args)
        return r.fingerprint(), int(r.stats[RESTARTS])

    print("[memory] free device", flush=True)
    want, fewest = run()
    assert fewest > 0
    total = torch.cuda.mem_get_info()[1]
    gc.collect()
    trim_memory()
    hold = torch.empty(_free() - total // 4 - 2048 * MB, dtype=torch.uint8, device="cuda")
    try:
        print("[memory] nothing kept", flush=True)
        got, alone = run()
        assert got == want and alone >= fewest
        print("[memory] blocks kept", flush=True)
        march(*workload("sphere"), table_log2=29)     # leaves a table of 2 GiB
        gc.collect()
        got, kept = run()
        print(f"[memory] restarts: {fewest} on a free device, {alone} nearly full, {kept} with blocks kept", flush=True)
        assert got == want and kept <= alone
    finally:
        del hold
        torch.cuda.empty_cache()
        gc.collect()
        trim_memory()
    assert abs(base - _free()) < 64 * MB
