"""A finer level's ghost cells are interpolated in time from the coarser
level's old state after its clean_state (CAMR_advance.cpp:83).  Levels that
step pass by pass clean it in place, and so do coarse levels with gravity on
either engine: states that clean_state changes (mass fractions that do not sum
to one to the last bit, or lie below zero) against the oracle's subcycled step,
bit for bit.  (A coarse level on the fused step cleans copies and leaves its
old state as it was; there the two differ by what clean_state changes.)"""
import numpy as np
import pytest

from camr_amd import _lib
from camr_amd.hydro import FluxRegister, amr_advance
from tests.test_gpu_amr import _pair
from tests.test_oracle_amr import FINE2, FINE3, _boxes

pytestmark = pytest.mark.gpu


def _with_species(U, lo, n, amp):
    """Three species of varying mass fractions; amp 1 takes one below 0."""
    k, j, i = np.meshgrid(*[np.arange(s) + l for s, l in zip(U.shape[1:], lo[::-1])], indexing="ij")
    s = 32 / n
    y0 = 0.5 + 0.2 * amp * np.sin(0.7 * i * s + 0.3 * j * s)
    y1 = 0.3 + 0.1 * amp * np.cos(0.5 * k * s + 0.2 * i * s)
    U = U.copy()
    U[7], U[8], U[9] = U[0] * y0, U[0] * y1, U[0] * (1.0 - y0 - y1)
    return U


@pytest.mark.parametrize("levels", [2, 3])
@pytest.mark.parametrize("amp", [0.5, 1.0])
@pytest.mark.parametrize("engine,grav", [(_lib.ENGINE_STAGED, 0.0), (_lib.ENGINE_STAGED, -0.9),
                                         (_lib.ENGINE_FUSED, -0.9)])
def test_ghosts_from_the_cleaned_old_state(oracle, levels, amp, engine, grav):
    print(f"old state: {levels} levels, amp {amp}, gravity {grav}, engine {engine}", flush=True)
    grids = [(16, _boxes(16, 8)), (32, FINE2), (64, FINE3)][:levels]
    pairs = [_pair(oracle, n, boxes, True, dict(ppm_type=1, const_grav=grav), engine=engine)
             for n, boxes in grids]
    for (n, boxes), pair in zip(grids, pairs):
        for b, bx in enumerate(boxes):
            U = _with_species(pair[0].get_box(b), bx[:3], n, amp)
            for L in pair:
                L.set_box(b, U)
    ol, gl = [p[0] for p in pairs], [p[1] for p in pairs]
    oR = [oracle.FluxRegister(ol[l], ol[l + 1], 2) for l in range(levels - 1)]
    gR = [FluxRegister(gl[l], gl[l + 1], 2) for l in range(levels - 1)]
    for l in reversed(range(levels - 1)):
        oracle.average_down(ol[l], ol[l + 1], 2)
        gl[l].average_down(gl[l + 1], 2)
    for L in ol + gl:
        L.init_post()
    dt = None
    for s in range(2):
        est = [[L.initial_dt() if s == 0 else L.new_dt(dt / 2 ** l) for l, L in enumerate(Ls)]
               for Ls in (ol, gl)]
        assert est[0] == est[1]
        dt = min(e * 2 ** l for l, e in enumerate(est[0]))
        assert oracle.amr_advance(ol, oR, dt) == 0
        amr_advance(gl, gR, dt)
        for l in range(levels):
            for b in range(len(ol[l].boxes)):
                assert np.array_equal(gl[l].get_box(b), ol[l].get_box(b)), (s, l, b)
    for r in gR + oR:
        r.close()
