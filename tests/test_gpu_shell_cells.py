"""The lists of coarse-fine ghost cells, made on the device: fine boxes in a
corner, across a periodic face, thinner than the ghost region, beside each
other and alone, with walls, ratios 2 and 4.  The oracle interpolates every
cell of the fine domain; a step on the listed cells alone equals it."""
import numpy as np
import pytest

from camr_amd import _lib, problems
from camr_amd.hydro import Level, Problem
from tests.test_gpu_parity import _oracle_params, assert_bitwise

pytestmark = pytest.mark.gpu

C = (12, 8, 10)  # coarse cells
BOXES = {"corner": [(0, 0, 0, 7, 7, 7)],
         "far_corner": [(16, 8, 12, 23, 15, 19)],
         "thin": [(9, 0, 6, 9, 15, 7)],
         "pair": [(4, 4, 4, 9, 11, 9), (10, 4, 4, 14, 11, 12)],
         "apart": [(1, 2, 3, 4, 6, 8), (15, 9, 11, 20, 13, 16)]}
CASES = [(name, bc, 2) for name in BOXES for bc in ((0, 0, 0), (2, 0, 4))
         if not (name == "thin" and bc[0])] + [("corner", (2, 2, 2), 2), ("pair", (0, 2, 0), 4)]


def _problem(n, boxes, bc, dx):
    return Problem(domlo=(0, 0, 0), domhi=tuple(x - 1 for x in n), dx=(dx,) * 3, bclo=bc, bchi=bc,
                   is_periodic=tuple(int(b == 0) for b in bc), boxes=boxes,
                   params=dict(ppm_type=1, cfl=0.4))


@pytest.mark.parametrize("name,bc,ratio", CASES)
@pytest.mark.parametrize("engine", [_lib.ENGINE_FUSED, _lib.ENGINE_STAGED])
def test_step_on_listed_ghosts(oracle, name, bc, ratio, engine):
    print(f"shell cells {name} bc {bc} ratio {ratio} engine {engine}", flush=True)
    n = tuple(x * ratio for x in C)
    coarse = _problem(C, [(0, 0, 0, 5, 7, 9), (6, 0, 0, 11, 7, 9)], bc, 1 / 12)
    fine = _problem(n, BOXES[name], bc, 1 / (12 * ratio))
    pairs = []
    for prob, m in ((coarse, 12), (fine, 12 * ratio)):
        full = problems.SmoothField(seed=3, kmax=2, mach=0.4).state(m, (0, 0, 0), prob.domhi)
        o = oracle.Level(_oracle_params(oracle, prob), prob.boxes)
        g = Level(prob, engine=engine)
        for L in (o, g):
            for b, x in enumerate(prob.boxes):
                L.set_box(b, np.ascontiguousarray(full[:, x[2]:x[5] + 1, x[1]:x[4] + 1,
                                                       x[0]:x[3] + 1]))
        if prob is coarse:
            o.init_post()
            g.init_post()
        pairs.append((o, g))
    (oc, gc), (of, gf) = pairs
    of.exterior_from_coarse(oc, ratio)
    gf.exterior_from_coarse(gc, ratio)
    of.init_post()
    gf.init_post()
    err, dts = of.run(2)
    assert err == 0
    assert np.array_equal(dts, gf.run(2))
    for b in range(len(fine.boxes)):
        assert_bitwise(gf.get_box(b), of.get_box(b), f"box {b}")
