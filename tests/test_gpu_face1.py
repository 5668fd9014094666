"""The traces and first fluxes in one kernel (k_face1_*), at the sizes where
its blocks can go wrong: rows shorter and longer than a tile's 16 cells,
a last tile of one face, rows that wrap inside a block, boxes of one cell,
PPM and PLM, with walls (the boundary states written back) and periodic;
whole level steps against the oracle, bit for bit."""
import numpy as np
import pytest

from camr_amd import workloads
from camr_amd.hydro import Level, Problem
from tests.test_gpu_parity import _oracle_params, assert_bitwise

pytestmark = pytest.mark.gpu

# grow(bx, 2) has n + 4 cells along a direction and n + 3 first faces: a
# tile of 16 cells holds 15 faces, so n = 12 is one whole tile, 13 leaves one
# face for a second, 27 and 28 the same one tile on
SHAPES = [(12, 13, 11), (13, 12, 28), (27, 5, 13), (4, 28, 5), (61, 4, 9)]
# a reflecting wall needs as many cells as there are ghosts
CASES = [(n, w) for n in SHAPES for w in (False, True)] + [((1, 1, 1), False), ((33, 1, 2), False)]


@pytest.mark.parametrize("ppm", [0, 1])
@pytest.mark.parametrize("n,walls", CASES)
def test_trace_and_first_flux_blocks(oracle, n, walls, ppm):
    print(f"face1 n={n} walls={walls} ppm={ppm}", flush=True)
    bc = (2, 4, 4) if walls else (0, 0, 0)
    prob = Problem(domlo=(0, 0, 0), domhi=tuple(x - 1 for x in n), dx=(1.0 / max(n),) * 3,
                   bclo=bc, bchi=bc, is_periodic=(0,) * 3 if walls else (1,) * 3,
                   boxes=[(0, 0, 0) + tuple(x - 1 for x in n)],
                   params=dict(ppm_type=ppm, cfl=0.3))
    U = workloads.smooth_field().state(max(max(n), 8), (0, 0, 0), tuple(x - 1 for x in n))
    o = oracle.Level(_oracle_params(oracle, prob), prob.boxes)
    g = Level(prob)
    for L in (o, g):
        L.set_box(0, U)
        L.init_post()
    err, od = o.run(2)
    assert err == 0
    gd = g.run(2)
    assert np.array_equal(od, gd)
    assert_bitwise(g.get_box(0), o.get_box(0), "state")
