"""What the operators refuse, and that they say so: the calls reach the PyTorch extension first, whose checks run in C++."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def _encoded(rows=64, K=256, S=4, G=128, L=16, seed=0):
    from sbvr import synth
    return [t.to(DEV) for t in synth.random_encoding(rows, K, S, G, L, seed=seed)]


def test_an_index_without_groups_is_an_error():
    """No group length given and no rows of indices to take it from: an exception in every operator (in C++ an integer
    division by zero would end the process)."""
    import sbvr
    from sbvr import _sbvr_hip_ops as ops
    none = torch.zeros(0, dtype=torch.float16, device=DEV)
    lb, li, lc = _encoded(2, seed=1)
    rb, ri, rc = _encoded(64, seed=2)
    x = torch.zeros((1, 256), dtype=torch.float16, device=DEV)
    with pytest.raises(ZeroDivisionError):
        sbvr._sbvr_mm_T(lb, li[:0], lc, rb, ri[:0], rc, none)
    with pytest.raises(RuntimeError, match="no groups"):
        ops._sbvr_mm_T(lb, li[:0], lc, rb, ri[:0], rc, none)
    tb, ti, tc = _encoded(256, 256, seed=3)
    with pytest.raises(ZeroDivisionError):
        sbvr._sbvr_row_deq_mm_T(x, tb, ti[:0], tc, none)
    with pytest.raises(RuntimeError, match="no groups"):
        ops._sbvr_row_deq_mm_T(x, tb, ti[:0], tc, none)
    with pytest.raises(ZeroDivisionError):
        sbvr._sbvr_linear_f16(x, rb, ri[:0], rc)
    with pytest.raises(RuntimeError, match="no groups"):
        ops._sbvr_linear_f16(x, rb, ri[:0], rc)
    with pytest.raises(RuntimeError):
        sbvr.SBVRLinear(256, 64, rb[:0], ri[:0], rc, 128)(x)


def test_the_operators_let_other_threads_run():
    """The products of encoded operands, the encoding on the fly and the decode release the interpreter's lock: with
    a switch interval that never ends, a second thread runs during these calls alone."""
    import sys
    import threading
    import time
    from sbvr import _sbvr_hip_ops as ops, synth
    none = torch.zeros(0, dtype=torch.float16, device=DEV)
    l, r, t = _encoded(2, seed=1), _encoded(64, seed=2), _encoded(256, 256, seed=3)
    x = torch.zeros((2, 256), dtype=torch.float16, device=DEV)
    lines = synth.make_lines(2, 4, 1.0, 7).to(DEV)
    calls = [lambda: ops._sbvr_mm_T(*l, *r, none), lambda: ops._sbvr_row_deq_mm_T(x, *t, none),
             lambda: ops._online_encode_lines(x, lines, 128), lambda: ops._decode_weight(*r, 128, 256, torch.float16)]
    ran, stop = [0], [False]

    def other():
        while not stop[0]:
            ran[0] += 1
            time.sleep(0)                # (gives the lock up, wants it back)

    for call in calls:
        call()
    torch.cuda.synchronize()
    interval = sys.getswitchinterval()
    thread = threading.Thread(target=other, daemon=True)
    try:
        sys.setswitchinterval(1000.0)
        thread.start()
        for call in calls:
            before = ran[0]
            for _ in range(500):
                call()
            assert ran[0] > before
    finally:
        sys.setswitchinterval(interval)
        stop[0] = True
        thread.join(10)
