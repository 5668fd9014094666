"""The method of lines' hydro source of a level (k_mol_xy, k_mol_z) where its
tiles can go wrong: boxes smaller than a tile's rim, rows, columns and planes
one past a tile, uneven boxes in one level, walls, slope orders and three
species; whole steps against the oracle, bit for bit."""
import numpy as np
import pytest

from camr_amd import problems
from camr_amd.hydro import Level, Problem
from tests.test_gpu_gravity import _species
from tests.test_gpu_parity import _oracle_params, assert_bitwise

pytestmark = pytest.mark.gpu

# one box of n cells: 18 x 14 tiles hold 16 x 12 cells of a plane, x-z tiles of
# 32 x 8 hold 32 x 6
ONE = [(4, 4, 4), (1, 5, 9), (16, 12, 6), (17, 13, 7), (33, 25, 18), (64, 4, 5), (70, 3, 2)]
CASES = [dict(n=n, bc=(0, 0, 0), order=4) for n in ONE] + [
    dict(n=(17, 13, 9), bc=(2, 4, 5), order=4), dict(n=(20, 9, 21), bc=(4, 5, 3), order=2),
    dict(n=(9, 16, 11), bc=(5, 2, 4), order=1)]


def _run(oracle, prob, full, steps=2):
    p = _oracle_params(oracle, prob)
    p.do_mol = 1
    p.plm_iorder = prob.value("plm_iorder")
    o, g = oracle.Level(p, prob.boxes), Level(prob)
    for L in (o, g):
        for b, x in enumerate(prob.boxes):
            L.set_box(b, np.ascontiguousarray(full[:, x[2]:x[5] + 1, x[1]:x[4] + 1, x[0]:x[3] + 1]))
        L.init_post()
    err, od = o.run(steps)
    assert err == 0
    assert np.array_equal(od, g.run(steps))
    for b in range(len(prob.boxes)):
        assert_bitwise(g.get_box(b), o.get_box(b), f"box {b}")


@pytest.mark.parametrize("case", CASES)
def test_one_box(oracle, case):
    n, bc = case["n"], case["bc"]
    print(f"MOL source {case}", flush=True)
    per = tuple(int(b == 0) for b in bc)
    prob = Problem(domlo=(0, 0, 0), domhi=tuple(x - 1 for x in n), dx=(1.0 / max(n),) * 3, bclo=bc,
                   bchi=bc, is_periodic=per, boxes=[(0, 0, 0) + tuple(x - 1 for x in n)],
                   params=dict(do_mol=1, cfl=0.3, plm_iorder=case["order"]))
    full = _species(problems.SmoothField(seed=7, kmax=3, mach=0.4).state(80, (0, 0, 0), prob.domhi))
    _run(oracle, prob, full)


def test_uneven_boxes(oracle):
    prob = Problem(domlo=(0, 0, 0), domhi=(39, 27, 18), dx=(1 / 40,) * 3, bclo=(2, 0, 4),
                   bchi=(4, 0, 2), is_periodic=(0, 1, 0),
                   boxes=[(0, 0, 0, 18, 27, 18), (19, 0, 0, 39, 12, 6), (19, 13, 0, 39, 27, 6),
                          (19, 0, 7, 39, 27, 18)],
                   params=dict(do_mol=1, cfl=0.3, const_grav=-0.7))
    full = _species(problems.SmoothField(seed=9, kmax=3, mach=0.4).state(40, (0, 0, 0), prob.domhi))
    _run(oracle, prob, full, 3)
