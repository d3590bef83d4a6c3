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


def test_errors_of_the_operators_keep_their_kinds():
    """What the extension refuses is refused by the checks in Python, each with its own kind of error."""
    import sbvr
    from sbvr import hip, synth
    none = torch.zeros(0, dtype=torch.float16, device=DEV)
    l, r, t = _encoded(2, seed=1), _encoded(64, seed=2), _encoded(256, 256, seed=3)
    x = torch.zeros((2, 256), dtype=torch.float16, device=DEV)
    lines = synth.make_lines(2, 4, 1.0, 7).to(DEV)
    longer = _encoded(64, 512, seed=4)
    strided = torch.zeros((2, 512), dtype=torch.float16, device=DEV)[:, ::2]

    def swapped(arrays, at, value):
        return [value if i == at else a for i, a in enumerate(arrays)]

    both = [*l, *r]
    for error, args in ((TypeError, swapped(both, 2, l[2].float())), (TypeError, swapped(both, 4, r[1].to(torch.int32).to(torch.uint16))),
                        (TypeError, swapped(both, 1, None)), (ValueError, [*l, *longer]), (ValueError, swapped(both, 5, r[2][0])),
                        (ValueError, swapped(both, 1, l[1].t())), (sbvr.hip.SbvrHipError, swapped(both, 3, r[0].cpu()))):
        with pytest.raises(error):
            sbvr._sbvr_mm_T(*args, none, bvr_len=128)
    with pytest.raises(ValueError):
        sbvr._sbvr_mm_T(*both, none, bvr_len=64)
    with pytest.raises(TypeError):
        sbvr._sbvr_mm_T(*both, torch.zeros(64, device=DEV), bvr_len=128)      # a bias of another type
    for error, args in ((TypeError, [x.float(), *t]), (ValueError, [strided, *t]), (ValueError, [x[:, :128].contiguous(), *t]),
                        (ValueError, [x[0], *t]), (sbvr.hip.SbvrHipError, [x.cpu(), *t])):
        with pytest.raises(error):
            sbvr._sbvr_row_deq_mm_T(*args, none, bvr_len=128)
    for error, args in ((TypeError, (x.float(), lines, 128)), (ValueError, (x, lines[:1], 128)), (ValueError, (strided, lines, 128)),
                        (hip.SbvrHipError, (x[:0], lines, 128)), (hip.SbvrHipError, (x.cpu(), lines, 128))):
        with pytest.raises(error):
            hip.online_encode_lines(*args)
    for error, args in ((TypeError, swapped(r, 2, r[2].float())), (ValueError, swapped(r, 1, r[1][:1])), (ValueError, swapped(r, 1, r[1].t())),
                        (hip.SbvrHipError, swapped(r, 0, r[0].cpu()))):
        with pytest.raises(error):
            hip.decode_weight(*args, 128, 256, torch.float16)
    with pytest.raises(hip.SbvrHipError):
        hip.decode_weight(*r, 128, 257, torch.float16)                        # more columns than there are
    # and everything still answers
    assert sbvr._sbvr_mm_T(*both, none, bvr_len=128).shape == (2, 64)
    assert hip.decode_weight(*r, 128, 256, torch.float16).shape == (64, 256)


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
            for _ in range(20000):           # (the waiting thread has to wake up while the lock is free)
                call()
                if ran[0] > before:
                    break
            assert ran[0] > before
    finally:
        sys.setswitchinterval(interval)
        stop[0] = True
        thread.join(10)
