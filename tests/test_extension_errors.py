"""Which errors of the PyTorch extension send a call on to the checks in Python, and which end it (no GPU: a stand-in
for the extension raises them)."""
import types

import pytest
import torch


class _Refused(RuntimeError):
    pass


class _LaunchFailed(RuntimeError):
    pass


def _calls():
    from sbvr import hip
    t = torch.zeros((4, 4), dtype=torch.float16)
    b = torch.zeros((4, 4, 4), dtype=torch.int32).view(torch.uint32)
    i = torch.zeros((1, 4), dtype=torch.uint8)
    return {"_sbvr_mm_T": lambda: hip._sbvr_mm_T(b, i, t, b, i, t, None), "_sbvr_row_deq_mm_T": lambda: hip._sbvr_row_deq_mm_T(t, b, i, t, None),
            "_online_encode_lines": lambda: hip.online_encode_lines(t, t, 32),
            "_decode_weight": lambda: hip.decode_weight(b, i, t, 128, 128, torch.float16)}


@pytest.mark.parametrize("name", ["_sbvr_mm_T", "_sbvr_row_deq_mm_T", "_online_encode_lines", "_decode_weight"])
def test_only_refused_arguments_go_on_to_the_checks_in_python(monkeypatch, name):
    from sbvr import hip
    made = []

    def stand_in(error):
        def op(*args):
            made.append(name)
            raise error
        return types.SimpleNamespace(Refused=_Refused, LaunchFailed=_LaunchFailed, **{name: op})

    call = _calls()[name]
    # refused, or arguments of another kind: the checks in Python give their own error (the tensors are not on a GPU)
    for error in (_Refused("shape"), TypeError("incompatible function arguments")):
        monkeypatch.setattr(hip, "_extension", stand_in(error))
        with pytest.raises(hip.SbvrHipError, match="GPU"):
            call()
    # the device or an allocation failed: reported as it is, the call is not made again
    for error, seen in ((_LaunchFailed("launch"), hip.SbvrHipError), (torch.OutOfMemoryError("memory"), torch.OutOfMemoryError),
                        (RuntimeError("device"), RuntimeError)):
        made.clear()
        monkeypatch.setattr(hip, "_extension", stand_in(error))
        with pytest.raises(seen, match=str(error)) as info:
            call()
        assert type(info.value) is seen and made == [name]


def test_the_extension_has_the_two_kinds_of_errors():
    from sbvr import _sbvr_hip_ops as ops
    assert issubclass(ops.Refused, RuntimeError) and issubclass(ops.LaunchFailed, RuntimeError)
    t = torch.zeros((4, 4), dtype=torch.float16)
    b = torch.zeros((4, 4, 4), dtype=torch.int32).view(torch.uint32)
    with pytest.raises(ops.Refused, match="must be on a GPU"):
        ops._decode_weight(b, t, t, 128, 128, torch.float16)
