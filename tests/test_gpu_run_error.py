"""A march that stops with an error leaves nothing running: the same context then marches on another stream,
with another network's weights, and gives a fresh context's records."""
import numpy as np
import pytest

from analyticmesh_amd import configs
from analyticmesh_amd.engine import Engine

pytestmark = pytest.mark.gpu


def _args(spec, n_seeds):
    p = configs.seeds_fibonacci(spec, n_seeds)
    w, b = ([np.asarray(a, np.float64) for a in arrays] for arrays in (spec.weights, spec.biases))
    return w, b, p, configs.mask_of(spec, p)


@pytest.mark.parametrize("precision", ["fp64", "fp64ray", "fp32"])
def test_run_on_another_stream_after_the_region_limit(precision):
    import torch
    nodes = [3, 64, 64, 1]
    a = _args(configs.geometric(nodes, 0.5, 0.03, 1), 24)
    b = _args(configs.geometric(nodes, 0.4, 0.05, 2), 24)
    want = Engine(nodes, precision=precision).run(*b)
    eng = Engine(nodes, precision=precision)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for turn, limit in enumerate([400, 1500, 4000]):
        print(f"[run error] {precision} limit {limit}", flush=True)
        eng.set_option("region_limit", limit)
        with pytest.raises(RuntimeError, match="am error 4"):
            eng.run(*a, stream=streams[turn % 2].cuda_stream)
        assert streams[turn % 2].query()          # nothing is left on the stream
        eng.set_option("region_limit", -1)
        got = eng.run(*b, stream=streams[1 - turn % 2].cuda_stream)
        for k in ("masks", "tabs", "vpairs", "verts"):
            assert np.array_equal(getattr(got, k), getattr(want, k)), (turn, k)
