"""The cut-cell stages in merged launches, at the box shapes where a launch's
entries end: against the oracle where the stages' list of (stage, box)
entries is flattened and where it is a two-dimensional grid, and against the
pair-by-pair launches (set_eb(merge=False)), which share one buffer among the
transverse pairs.  Bit for bit.
"""
import numpy as np
import pytest

from camr_amd import _lib, workloads
from camr_amd.hydro import Level
from test_gpu_eb import _oracle_params

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _level(prob, geom, merge=True):
    L = Level(prob, engine=_lib.ENGINE_STAGED)
    L.set_eb(geom, merge=merge)
    for b in range(len(prob.boxes)):
        L.set_box(b, workloads.sod_sphere_init(prob, b, geom))
    L.init_post()
    return L


# cut-cell boxes: one of 48x24x24; with a remainder at the high faces; more
# entries (stages * boxes) than a launch holds flattened; more cut cells than
# the divergence takes a component at a time
@pytest.mark.parametrize("n,max_grid,steps", [(24, 48, 3), (24, 10, 3), (24, 6, 3), (96, 32, 1)])
def test_merged_stages_match_oracle_and_pair_by_pair(oracle, n, max_grid, steps):
    print(f"EB stages: n={n} max_grid={max_grid}", flush=True)
    prob = workloads.sod_sphere(n=n, max_grid=max_grid, interface=0.4)
    geom = workloads.sod_sphere_geometry(prob)
    A, B = _level(prob, geom), _level(prob, geom, merge=False)
    assert 1 in A.kinds
    ol = oracle.Level(_oracle_params(oracle, prob), prob.boxes)
    ol.set_eb(geom)
    for b in range(len(prob.boxes)):
        ol.set_box(b, workloads.sod_sphere_init(prob, b, geom))
    ol.init_post()
    err, odts = ol.run(steps)
    assert err == 0
    for L in (A, B):
        assert np.array_equal(np.asarray(L.run(steps)), odts)
        for b in range(len(prob.boxes)):
            assert np.array_equal(L.get_box(b), ol.get_box(b)), b
