"""What calls share behind the handles: kept device blocks beside another thread's stream capture."""
import ctypes as C
import threading

import numpy as np
import pytest

from votca_amd import pyxtp as px

pytestmark = pytest.mark.gpu


def tensor(o, v, P, seed, scale=0.1):
    rng = np.random.default_rng(seed)
    n = o + v
    M = rng.normal(scale=scale, size=(n, n, P))
    M = 0.5 * (M + M.transpose(1, 0, 2))
    e = np.concatenate([np.sort(rng.uniform(-1, -0.3, o)), np.sort(rng.uniform(0.1, 2.0, v))])
    return px.TCMatrix_gwbse().Initialize(P, 0, n - 1, 0, n - 1).set_tensor(M), e, rng


def operator(t, e, eps, o, c=(1, 2, 1, 0)):
    return px.BSE_OPERATOR(*c, eps, t, np.diag(e)).configure(px.BSEOperator_Options(o - 1, 0, 0, 0, e.size - 1))


@pytest.mark.parametrize("mode", [1, 2])  # hipStreamCaptureModeThreadLocal, hipStreamCaptureModeRelaxed
def test_destroy_beside_another_threads_capture(mode):
    t, e, rng = tensor(24, 160, 200, 1)
    op = operator(t, e, rng.uniform(0.3, 1.0, 200), 24)  # M_cc' of 200 x 160 x 192: 49 MB, a kept block
    op.matmul(rng.normal(size=(op.size, 2)))
    hip = C.CDLL("libamdhip64.so")
    st, graph, status = C.c_void_p(), C.c_void_p(), C.c_int()
    assert hip.hipStreamCreateWithFlags(C.byref(st), 1) == 0
    assert hip.hipStreamBeginCapture(st, mode) == 0
    th = threading.Thread(target=op.close)
    th.start()
    th.join()
    assert hip.hipStreamIsCapturing(st, C.byref(status)) == 0
    end = hip.hipStreamEndCapture(st, C.byref(graph))
    assert status.value == 1 and end == 0  # still active, and a graph
    assert hip.hipGraphDestroy(graph) == 0 and hip.hipStreamDestroy(st) == 0
