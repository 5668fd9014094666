"""A level with constant gravity on the fused engine's step (the source
predictors come out of the ghost fill) against the oracle, bit for bit:
three species, walls and periodic sides, coarse-fine ghosts from exterior
data, batched and per box, the staged and the CTU transverse kernels, PLM
with the hydrostatic pressure slope, and density floors (the step repeated
pass by pass)."""
import numpy as np
import pytest

from camr_amd import _lib, problems, workloads
from camr_amd.hydro import Level, Problem
from tests.test_gpu_parity import _oracle_params, assert_bitwise

pytestmark = pytest.mark.gpu


def _species(U):
    """Three species of unequal, varying mass fractions."""
    k, j, i = np.meshgrid(*[np.arange(s) for s in U.shape[1:]], indexing="ij")
    y0 = 0.5 + 0.2 * np.sin(0.7 * i + 0.3 * j)
    y1 = 0.3 + 0.1 * np.cos(0.5 * k + 0.2 * i)
    U = U.copy()
    U[7], U[8], U[9] = U[0] * y0, U[0] * y1, U[0] * (1.0 - y0 - y1)
    return U


def _check(oracle, prob, full, steps, ext=None, batched=True, ctu=0, small_dens=None):
    p = _oracle_params(oracle, prob)
    if small_dens:
        p.small_dens = small_dens
    o = oracle.Level(p, prob.boxes)
    g = Level(prob, engine=_lib.ENGINE_FUSED, batched=batched)
    g.ctu = (ctu, 4)
    for L in (o, g):
        if ext is not None:
            L.set_exterior(ext)
        for b, x in enumerate(prob.boxes):
            L.set_box(b, np.ascontiguousarray(full[:, x[2]:x[5] + 1, x[1]:x[4] + 1, x[0]:x[3] + 1]))
        L.init_post()
    err, od = o.run(steps)
    assert err == 0
    assert np.array_equal(od, g.run(steps))
    for b in range(len(prob.boxes)):
        assert_bitwise(g.get_box(b), o.get_box(b), f"box {b}")


@pytest.mark.parametrize("ppm,pslope", [(1, 0), (0, 0), (0, 1)])
@pytest.mark.parametrize("batched,ctu", [(True, 0), (False, 0), (True, 1)])
def test_gravity_walls_and_periodic(oracle, ppm, pslope, batched, ctu):
    print(f"gravity ppm={ppm} pslope={pslope} batched={batched} ctu={ctu}", flush=True)
    prob = Problem(domlo=(0, 0, 0), domhi=(18, 13, 15), dx=(1 / 19,) * 3, bclo=(2, 0, 4),
                   bchi=(4, 0, 5), is_periodic=(0, 1, 0),
                   boxes=[(0, 0, 0, 10, 13, 15), (11, 0, 0, 18, 13, 15)],
                   params=dict(ppm_type=ppm, cfl=0.4, const_grav=-1.3, use_pslope=pslope))
    full = _species(problems.SmoothField(seed=5, kmax=3, mach=0.4).state(32, (0, 0, 0), (18, 13, 15)))
    _check(oracle, prob, full, 3, batched=batched, ctu=ctu)


def test_gravity_with_exterior(oracle):
    prob = workloads.refined_level(n=32, radius=0.3, blocking_factor=8, max_size=16)
    prob.params["const_grav"] = 0.8
    full = _species(workloads.exterior(prob))
    _check(oracle, prob, full, 2, ext=full)


def test_gravity_with_density_floors(oracle):
    prob = workloads.smooth_periodic(n=16, ppm_type=1, max_grid=8)
    prob.params.update(small_dens=0.95, const_grav=-0.7)
    full = workloads.smooth_field().state(16)
    _check(oracle, prob, full, 3, small_dens=0.95)
