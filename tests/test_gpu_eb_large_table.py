"""Cut-cell boxes whose stages are more than kStageMergeBlocks blocks: a
launch per stage, with a buffer per transverse pair.  Forward against the
oracle and the pair-by-pair launches (set_eb(merge=False)) bit for bit; the
gradient of the force against the pair-by-pair one, whose sums go in another
order (atomics: the same run twice differs by 2e-16 of the norm and 8e-15 in
one entry)."""
import numpy as np
import pytest

from camr_amd import _lib, workloads
from camr_amd.hydro import Level
from test_gpu_eb import _oracle_params

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

N = 128  # one box of 256 x 128 x 128: three faces of the box alone are 49347 blocks


@pytest.fixture(scope="module")
def grid():
    prob = workloads.sod_sphere(n=N, max_grid=2 * N, interface=0.4)
    assert len(prob.boxes) == 1
    return prob, workloads.sod_sphere_geometry(prob)


def _level(prob, geom, merge, init):
    L = Level(prob, engine=_lib.ENGINE_STAGED)
    L.set_eb(geom, merge=merge)
    assert list(L.kinds) == [1]
    L.set_box(0, init(prob, 0, geom))
    L.init_post()
    return L


def _launches(L, what, run):
    """Launches of the cut-cell stages named what* while run() works."""
    L.profile(True)
    run()
    rep = L.profile_report()
    L.profile(False)
    return sum(r["count"] for k, r in rep.items() if k.startswith(what))


def test_step(oracle, grid):
    prob, geom = grid
    print("cut cells, a launch per stage: step", flush=True)
    A, B = (_level(prob, geom, m, workloads.sod_sphere_init) for m in (True, False))
    o = oracle.Level(_oracle_params(oracle, prob), prob.boxes)
    o.set_eb(geom)
    o.set_box(0, workloads.sod_sphere_init(prob, 0, geom))
    o.init_post()
    err, od = o.run(1)
    assert err == 0
    for L in (A, B):
        assert np.array_equal(np.asarray(L.run(1)), od)
        assert np.array_equal(L.get_box(0), o.get_box(0))
    assert _launches(A, "eb_", lambda: A.run(1)) == 32  # 31 stages and the primitives


def test_gradient(grid):
    prob, geom = grid
    print("cut cells, a launch per stage: gradient", flush=True)
    grads = []
    for merge in (True, False):
        L = _level(prob, geom, merge, workloads.sod_sphere_smooth_init)

        def gradient():
            L.adjoint_forward([2e-3] * 2, 1)
            L.seed_force_adjoint((1.0, 0.3, -0.2))
            L.adjoint_backward()

        assert _launches(L, "ebadj_", gradient) == 2 * 31
        grads.append(L.get_adjoint(0))
        L.close()
    a, b = grads
    d = np.abs(a - b)
    assert np.linalg.norm(b) > 0.0
    assert np.linalg.norm(d) <= 3e-15 * np.linalg.norm(b)
    rms = np.sqrt((b ** 2).mean())
    assert (d <= 1e-12 * np.maximum(np.abs(b), rms)).all()
