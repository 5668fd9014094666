"""hydro_umdrv with flux arrays that are not three dense ones apart from each
other: dS/dt does not depend on how the caller lays the fluxes out, nor on
whether they share memory; the fluxes are right wherever no two share an
element.  Against a call with three separate arrays, bit for bit."""
import ctypes as C

import pytest

from camr_amd import _lib
from camr_amd.hydro import Problem, _box, array4_of, hydro_ctoprim, hydro_params

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from tests.test_gpu_parity import _box_state  # noqa: E402

LO, HI = (2, -1, 3), (14, 6, 11)
N = tuple(h - l + 1 for l, h in zip(LO, HI))
# faces per direction, x first
FACES = [tuple(N[a] + (a == d) for a in range(3)) for d in range(3)]


def _view(buf, first, strides, d):
    """Array4 of the d-faces: element (lo, 0) is buf[first], strides (j, k, n)."""
    a = _lib.Array4()
    a.p = buf.data_ptr() + 8 * first
    a.jstride, a.kstride, a.nstride = strides
    for x in range(3):
        a.lo[x], a.hi[x] = LO[x], HI[x] + (x == d)
    a.ncomp = 10
    return a


def _views(layout):
    """(buffers, their Array4s, tensors of the fluxes or None where they share
    elements)."""
    n = [f[0] * f[1] * f[2] for f in FACES]
    if layout == "interleaved":  # one component of every direction after the other
        buf = torch.full((10, sum(n)), -7.0, dtype=torch.float64, device="cuda")
        at = [0, n[0], n[0] + n[1]]
        v = [_view(buf, at[d], (FACES[d][0], FACES[d][0] * FACES[d][1], sum(n)), d) for d in range(3)]
        t = [buf[:, at[d]:at[d] + n[d]].view(10, *FACES[d][::-1]) for d in range(3)]
        return [buf], v, t
    if layout == "component_inside":  # components between the rows
        bufs = [torch.full((f[2], f[1], 10, f[0]), -7.0, dtype=torch.float64, device="cuda")
                for f in FACES]
        v = [_view(b, 0, (10 * f[0], 10 * f[0] * f[1], f[0]), d)
             for d, (b, f) in enumerate(zip(bufs, FACES))]
        return bufs, v, [b.permute(2, 0, 1, 3) for b in bufs]
    buf = torch.full((10 * max(n),), -7.0, dtype=torch.float64, device="cuda")
    ns = [0 if layout == "one_plane" else m for m in n]
    bufs = [torch.full_like(buf, -7.0) for _ in range(3)] if layout == "one_plane" else [buf] * 3
    v = [_view(bufs[d], 0, (FACES[d][0], FACES[d][0] * FACES[d][1], ns[d]), d) for d in range(3)]
    return bufs, v, None


@pytest.mark.parametrize("layout", ["one_buffer", "one_plane", "interleaved", "component_inside"])
@pytest.mark.parametrize("ppm", [0, 1])
def test_flux_layouts(layout, ppm):
    print(f"flux layout {layout} ppm={ppm}", flush=True)
    prob = Problem(domlo=LO, domhi=HI, dx=(1 / 16,) * 3, bclo=(2, 0, 4), bchi=(4, 0, 2),
                   is_periodic=(0, 1, 0), boxes=[LO + HI], params=dict(ppm_type=ppm))
    hp = hydro_params(prob)
    glo, ghi = tuple(x - 4 for x in LO), tuple(x + 4 for x in HI)
    U = torch.from_numpy(_box_state(glo, ghi, seed=5)).cuda()
    q = torch.zeros((11,) + U.shape[1:], dtype=torch.float64, device="cuda")
    qa = torch.zeros((5,) + U.shape[1:], dtype=torch.float64, device="cuda")
    hydro_ctoprim(glo, ghi, U, glo, q, qa, hp)

    def call(views):
        ds = torch.zeros((10,) + N[::-1], dtype=torch.float64, device="cuda")
        none = _lib.Array4()
        _lib.check(_lib.lib().camr_hydro_umdrv(
            C.byref(_box(LO, HI)), C.byref(array4_of(U, glo)), C.byref(array4_of(ds, LO)),
            C.byref(array4_of(q, glo)), C.byref(array4_of(qa, glo)), C.byref(none),
            (_lib.Array4 * 3)(*views), (_lib.Array4 * 3)(none, none, none), C.byref(none),
            0.02, C.byref(hp), None))
        torch.cuda.synchronize()
        return ds

    ref = [torch.zeros((10,) + f[::-1], dtype=torch.float64, device="cuda") for f in FACES]
    want = call([array4_of(f, LO) for f in ref])
    bufs, views, fluxes = _views(layout)
    assert torch.equal(call(views), want)
    for d in range(3 if fluxes else 0):
        assert torch.equal(fluxes[d], ref[d]), d
