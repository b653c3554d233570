"""What calls share behind the handles: kept device blocks beside another thread's stream capture, and the scratch
of one context between threads."""
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


def test_threads_share_a_context_scratch():
    """The self-energy, the adjoint and the diagonal of a new operator, two threads each on one context and at
    different sizes, give the bits that they give alone."""
    calls = []
    for o, v, P, per in ((5, 37, 70, 2), (9, 83, 130, 5)):
        t, e, rng = tensor(o, v, P, P, 0.05)
        rpa = px.RPA(t)
        rpa.configure(o - 1, 0, e.size - 1)
        s = px.Sigma_PPM(t, rpa).configure(o - 1, 0, o + 3, 0, e.size - 1)
        s.ppm_weight, s.ppm_freq = rng.uniform(0, 0.5, P), rng.uniform(0.5, 2.0, P)
        s.set_rpa_energies(e)
        lv = np.repeat(np.arange(o + 4), per)
        om = rng.uniform(-2, 2, lv.size)
        eps = rng.uniform(0.3, 1.0, P)
        A, B = operator(t, e, eps, o), operator(t, e, eps, o, (0, 2, 0, 1))
        x, y = rng.normal(size=(o * v, 3)), rng.normal(size=(o * v, 3))

        def create(t=t, e=e, eps=eps, o=o):
            op = operator(t, e, eps, o)
            d = op.diagonal()
            op.close()
            return (d,)

        calls += [lambda s=s, lv=lv, om=om: s.diag_batch(lv, om),
                  lambda A=A, B=B, x=x, y=y: px.bse_adjoint(A, x, B, y), create]
    want = [[np.array(a) for a in c()] for c in calls]
    bad = []

    def work(i):
        for _ in range(15):
            if not all(np.array_equal(a, b) for a, b in zip(calls[i](), want[i])):
                bad.append(i)

    th = [threading.Thread(target=work, args=(i,)) for i in range(len(calls))]
    [x.start() for x in th]
    [x.join() for x in th]
    assert not bad
