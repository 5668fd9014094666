"""Which transverse kernels a level runs: one launch of all three directions
on small levels, and a launch per direction with the marching z kernels
wherever the caller sets a z-march, at any size.  The launches are counted by
the level's profiler; results against the oracle, bit for bit."""
import numpy as np
import pytest

from camr_amd import _lib, problems
from camr_amd.hydro import Level, Problem
from tests.test_gpu_gravity import _species
from tests.test_gpu_parity import _oracle_params, assert_bitwise

pytestmark = pytest.mark.gpu

BOXES = [(0, 0, 0, 10, 9, 12), (11, 0, 0, 18, 9, 12)]


def _problem(ppm, grav=0.0, **kw):
    return Problem(domlo=(0, 0, 0), domhi=(18, 9, 12), dx=(1 / 19,) * 3, bclo=(2, 0, 4),
                   bchi=(4, 0, 2), is_periodic=(0, 1, 0), boxes=BOXES,
                   params=dict(ppm_type=ppm, cfl=0.3, const_grav=grav, **kw))


def _march(planes):
    z = [0] * _lib.NSTAGE
    z[7] = z[11] = planes
    return z


def _launches(L):
    """Launches of the two transverse stages in one step, per box group."""
    L.profile(True)
    L.run(1)
    rep = L.profile_report()
    L.profile(False)
    return rep["transverse_1"]["count"], rep["transverse_2"]["count"]


@pytest.mark.parametrize("batched", [True, False])
def test_route(batched):
    full = problems.SmoothField(seed=3, kmax=3, mach=0.4).state(32, (0, 0, 0), (18, 9, 12))
    L = Level(_problem(1), batched=batched)
    for b, x in enumerate(BOXES):
        L.set_box(b, np.ascontiguousarray(full[:, x[2]:x[5] + 1, x[1]:x[4] + 1, x[0]:x[3] + 1]))
    L.init_post()
    n = 1 if batched else len(BOXES)
    assert _launches(L) == (n, n)
    for planes in (1, 2, 64):
        L.zmarch = _march(planes)
        assert L.zmarch == _march(planes)
        assert _launches(L) == (3 * n, 3 * n)
    z = _march(0)
    z[11] = 4
    L.zmarch = z
    assert _launches(L) == (n, 3 * n)
    L.zmarch = _march(0)
    assert _launches(L) == (n, n)
    L.zmarch = _march(3)
    L.tuning = L.tuning  # back to the defaults, which march on large levels only
    assert L.zmarch == _march(2)
    assert _launches(L) == (n, n)


# floors: the step is redone pass by pass, where the transdd kernels read
# every source component
@pytest.mark.parametrize("planes", [1, 5, 64])
@pytest.mark.parametrize("ppm,grav,floors", [(0, 0.0, False), (0, -1.3, False), (1, -1.3, True)])
@pytest.mark.parametrize("batched,graph", [(True, False), (False, False), (True, True)])
def test_marched_step_matches_oracle(oracle, planes, ppm, grav, floors, batched, graph):
    print(f"z-march {planes} ppm={ppm} grav={grav} floors={floors} batched={batched} graph={graph}",
          flush=True)
    prob = _problem(ppm, grav, **(dict(small_dens=0.95) if floors else {}))
    p = _oracle_params(oracle, prob)
    full = _species(problems.SmoothField(seed=8, kmax=3, mach=0.4).state(32, (0, 0, 0), (18, 9, 12)))
    if floors:
        p.small_dens = 0.95
        assert full[0].min() < 0.95
    o = oracle.Level(p, BOXES)
    g = Level(prob, batched=batched, graph=graph)
    g.zmarch = _march(planes)
    for L in (o, g):
        for b, x in enumerate(BOXES):
            L.set_box(b, np.ascontiguousarray(full[:, x[2]:x[5] + 1, x[1]:x[4] + 1, x[0]:x[3] + 1]))
        L.init_post()
    err, od = o.run(3)
    assert err == 0
    assert np.array_equal(od, g.run(3))
    for b in range(len(BOXES)):
        assert_bitwise(g.get_box(b), o.get_box(b), f"box {b}")
