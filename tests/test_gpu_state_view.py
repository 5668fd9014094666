"""The device view of a level's state after a step that a density floor has
the level redo: the redone one, taken right after the step on levels with
gravity and on the staged engine, after a sync on any level; an error of the
step reaches the caller."""
import numpy as np
import pytest

from camr_amd import _lib, workloads
from camr_amd.hydro import Level
from tests.test_gpu_parity import _oracle_params, assert_bitwise

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


class _Memory:
    def __init__(self, level, b):
        self.level = level
        self.__cuda_array_interface__ = {"shape": level.shape(b), "typestr": "<f8",
                                         "data": (level.state_array(b).p, False), "version": 3}


def _view(level, b):
    return torch.as_tensor(_Memory(level, b), device="cuda")


@pytest.mark.parametrize("engine,grav,sync", [(_lib.ENGINE_FUSED, -0.7, False), (_lib.ENGINE_STAGED, -0.7, False),
                                              (_lib.ENGINE_STAGED, 0.0, False), (_lib.ENGINE_FUSED, 0.0, True),
                                              (_lib.ENGINE_FUSED, -0.7, True)])
def test_view_after_a_floored_step(oracle, engine, grav, sync):
    print(f"state view: gravity {grav} engine {engine} sync {sync}", flush=True)
    prob = workloads.smooth_periodic(n=16, ppm_type=1, max_grid=8)
    prob.params.update(small_dens=0.95, const_grav=grav)
    p = _oracle_params(oracle, prob)
    p.small_dens = 0.95
    full = workloads.smooth_field().state(16)
    assert full[0].min() < 0.95 < full[0].max()
    o, g = oracle.Level(p, prob.boxes), Level(prob, engine=engine)
    for L in (o, g):
        for b, x in enumerate(prob.boxes):
            L.set_box(b, np.ascontiguousarray(full[:, x[2]:x[5] + 1, x[1]:x[4] + 1, x[0]:x[3] + 1]))
        L.init_post()
    for _ in range(2):
        assert o.advance(1e-3) == 0
        g.advance(1e-3)
        if sync:
            g.sync()
        got = [_view(g, b).cpu().numpy() for b in range(len(prob.boxes))]
        for b in range(len(prob.boxes)):
            assert_bitwise(got[b], o.get_box(b), f"box {b}")


def test_view_after_a_failed_step():
    prob = workloads.smooth_periodic(n=16, ppm_type=1)
    prob.params["const_grav"] = -0.7
    L = Level(prob, engine=_lib.ENGINE_FUSED)
    U = workloads.smooth_init(prob, 0)
    L.set_box(0, U)
    L.init_post()
    v = _view(L, 0)
    v[0, 3, 4, 5] = 0.0  # density zero: enforce_minimum_density aborts
    torch.cuda.synchronize()
    with pytest.raises(_lib.CamrError) as e:
        L.advance(1e-3)
        L.state_array(0)
    assert e.value.code == _lib.ERR_ZERO_DENSITY
    L.state_array(0)  # reported once
