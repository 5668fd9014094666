"""The kept status and result words of the synchronous per-box calls: a
failing hydro_ctoprim does not reach the next call's result, estdt calls
between them return their own minimum, and calls from several threads on
streams of their own see their own words."""
import threading

import numpy as np
import pytest

from camr_amd import _lib
from camr_amd.hydro import Problem, estdt_hydro, hydro_ctoprim, hydro_params

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from tests.test_gpu_parity import _box_state  # noqa: E402

LO, HI = (0, 0, 0), (8, 6, 4)


def _problem():
    return Problem(domlo=LO, domhi=HI, dx=(1 / 16,) * 3, bclo=(0,) * 3, bchi=(0,) * 3,
                   is_periodic=(1, 1, 1), boxes=[LO + HI])


def _calls(seed, bad, out):
    hp = hydro_params(_problem())
    U = torch.from_numpy(_box_state(LO, HI, seed=seed)).cuda()
    if bad:
        U[4] = -1.0
    q = torch.zeros((11,) + U.shape[1:], dtype=torch.float64, device="cuda")
    qa = torch.zeros((5,) + U.shape[1:], dtype=torch.float64, device="cuda")
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    for _ in range(20):
        try:
            hydro_ctoprim(LO, HI, U, LO, q, qa, hp, stream=s.cuda_stream)
            out.append(("ok", estdt_hydro(LO, HI, U, LO, (1 / 16,) * 3, stream=s.cuda_stream)))
        except _lib.CamrError:
            out.append(("refused", None))


def test_words_belong_to_one_call():
    ref = {}
    for seed in (1, 2):
        U = _box_state(LO, HI, seed=seed)
        c = np.sqrt(1.4 * 0.4 * U[5] / U[0])
        ref[seed] = min((1 / 16 / (c + np.abs(U[1 + d] / U[0]))).min() for d in range(3))
    outs = [[] for _ in range(4)]
    jobs = [(1, False), (1, True), (2, False), (2, True)]
    _calls(1, True, [])
    ts = [threading.Thread(target=_calls, args=(s, b, o)) for (s, b), o in zip(jobs, outs)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for (seed, bad), o in zip(jobs, outs):
        assert len(o) == 20
        for what, dt in o:
            assert what == ("refused" if bad else "ok")
            # three roundings apart from the kernel's operation order
            assert bad or abs(dt - ref[seed]) <= 8 * 2.3e-16 * ref[seed]
