"""The synchronous per-box calls beside a stream capture of another thread:
whatever they return, they leave that capture valid, also where a call fails
and its kept status word is cleared again."""
import ctypes as C
import threading

import pytest

from camr_amd.hydro import estdt_hydro, hydro_ctoprim, hydro_params
from tests.test_gpu_call_words import HI, LO, _problem

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from tests.test_gpu_parity import _box_state  # noqa: E402

THREAD_LOCAL = 1


def _hip():
    """The HIP runtime this process has loaded."""
    with open("/proc/self/maps") as f:
        return C.CDLL(next(x.split()[-1] for x in f if "libamdhip64" in x))


def _calls(fields, stream, out):
    hp = hydro_params(_problem())
    for U, q, qa in fields:
        try:
            hydro_ctoprim(LO, HI, U, LO, q, qa, hp, stream=stream.cuda_stream)
            out.append(estdt_hydro(LO, HI, U, LO, (1 / 16,) * 3, stream=stream.cuda_stream))
        except Exception as e:
            out.append(str(e))


def test_capture_of_another_thread_stays_valid():
    fields = []
    for bad in (False, True, False):
        U = torch.from_numpy(_box_state(LO, HI, seed=4)).cuda()
        if bad:
            U[4] = -1.0
        fields.append((U, *[torch.zeros((n,) + U.shape[1:], dtype=torch.float64, device="cuda")
                            for n in (11, 5)]))
    own = torch.cuda.Stream()
    torch.cuda.synchronize()
    hip, st, graph = _hip(), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreate(C.byref(st)) == 0  # waits for the null stream, and it for this
    plain, beside = [], []
    assert hip.hipStreamBeginCapture(st, THREAD_LOCAL) == 0
    t = threading.Thread(target=_calls, args=(fields, own, beside))
    t.start()
    t.join()
    assert hip.hipStreamEndCapture(st, C.byref(graph)) == 0
    assert hip.hipGraphDestroy(graph) == 0 and hip.hipStreamDestroy(st) == 0
    _calls(fields, own, plain)
    print(plain, beside, flush=True)
    assert isinstance(plain[0], float) and isinstance(plain[1], str) and plain[0] == plain[2]
    assert beside == plain
