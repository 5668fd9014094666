"""Subcycled hierarchies with constant gravity against the oracle, bit for
bit.  A level with a finer one steps pass by pass there (the finer level's
ghost cells are interpolated in time from its cleaned old state), the finest
level takes the fused step with its own gravity kernels, whose fluxes feed
the register, and which a density floor has redone between register adds."""
import numpy as np
import pytest

from camr_amd import _lib
from camr_amd.hydro import FluxRegister, amr_advance
from tests.test_gpu_amr import FACE, FINE4, _pair
from tests.test_oracle_amr import FINE2, FINE3, _boxes

pytestmark = pytest.mark.gpu

GRAV = -0.9


def _below_floor(L):
    """Box 0's state with two neighbouring cells below small_dens (1e-7)."""
    U = L.get_box(0)
    for i, rho in ((1, 5e-8), (2, 2e-8)):
        f = rho / U[0, 1, 1, i]
        U[[0, 1, 2, 3, 5, 7, 8, 9], 1, 1, i] *= f
        U[4, 1, 1, i] = U[5, 1, 1, i] + 0.5 * (U[1:4, 1, 1, i] ** 2).sum() / U[0, 1, 1, i]
    return U


def _run(oracle, grids, ratios, periodic, kw, engine, floors=(), steps=3):
    pairs = [_pair(oracle, n, boxes, periodic, dict(kw, const_grav=GRAV), engine=engine)
             for n, boxes in grids]
    for l in floors:
        U = _below_floor(pairs[l][0])
        for L in pairs[l]:
            L.set_box(0, U)
    ol, gl = [p[0] for p in pairs], [p[1] for p in pairs]
    oR = [oracle.FluxRegister(ol[l], ol[l + 1], r) for l, r in enumerate(ratios)]
    gR = [FluxRegister(gl[l], gl[l + 1], r) for l, r in enumerate(ratios)]
    for l in reversed(range(len(ratios))):
        oracle.average_down(ol[l], ol[l + 1], ratios[l])
        gl[l].average_down(gl[l + 1], ratios[l])
    for L in ol + gl:
        L.init_post()
    sub = [int(np.prod(ratios[:l])) for l in range(len(gl))]  # steps per coarse step
    dt = None
    for s in range(steps):
        est = [[L.initial_dt() if s == 0 else L.new_dt(dt / m) for L, m in zip(Ls, sub)]
               for Ls in (ol, gl)]
        assert est[0] == est[1], s
        dt = min(e * m for e, m in zip(est[0], sub))
        assert oracle.amr_advance(ol, oR, dt) == 0
        amr_advance(gl, gR, dt)
        for l in range(len(gl)):
            for b in range(len(ol[l].boxes)):
                assert np.array_equal(gl[l].get_box(b), ol[l].get_box(b)), (s, l, b)
    for r in gR + oR:
        r.close()


ENGINES = [_lib.ENGINE_FUSED, _lib.ENGINE_STAGED]


@pytest.mark.parametrize("ratio,periodic,ppm,face", [(2, True, 1, 0), (2, False, 0, 0), (4, True, 0, 0),
                                                     (4, False, 1, 0), (2, False, 1, 1), (4, True, 1, 1)])
@pytest.mark.parametrize("engine", ENGINES)
def test_two_levels(oracle, ratio, periodic, ppm, face, engine):
    print(f"two levels, gravity: ratio {ratio} periodic {periodic} ppm {ppm} face {face} "
          f"engine {engine}", flush=True)
    fine = FACE[ratio] if face else FINE2 if ratio == 2 else FINE4
    _run(oracle, [(16, _boxes(16, 8)), (16 * ratio, fine)], [ratio], periodic, dict(ppm_type=ppm), engine)


@pytest.mark.parametrize("ppm", [0, 1])
@pytest.mark.parametrize("engine", ENGINES)
def test_three_levels(oracle, ppm, engine):
    print(f"three levels, gravity: ppm {ppm} engine {engine}", flush=True)
    _run(oracle, [(16, _boxes(16, 8)), (32, FINE2), (64, FINE3)], [2, 2], True, dict(ppm_type=ppm),
         engine, steps=2)


@pytest.mark.parametrize("floors", [(1,), (0, 1)])
@pytest.mark.parametrize("engine", ENGINES)
def test_density_floor_between_register_adds(oracle, floors, engine):
    print(f"floors on levels {floors}, gravity: engine {engine}", flush=True)
    _run(oracle, [(16, _boxes(16, 8)), (32, FINE2)], [2], True, dict(ppm_type=0), engine, floors, steps=2)
