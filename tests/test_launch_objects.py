"""What launch_lowered takes as a lowered kernel and as buffers: any object with the four fields that it
reads, and any container that knows its names.  CPU: the entry point and the device checks are stubs."""

from collections import namedtuple
from types import SimpleNamespace

import pytest

from intent_ir_amd import launch_lowered, lower_intent_to_hip_kernel, runtime
from intent_ir_amd.configs import softmax_inner_ir

FIELDS = ("io_spec", "bindings", "call_args", "kernel_id")


@pytest.fixture
def calls(monkeypatch):
    """The arguments of each call that reaches the entry point."""
    import torch

    got = []
    lib = SimpleNamespace(**{n: (lambda *a: got.append(a) or 0) for n in runtime.SIGNATURES})
    monkeypatch.setattr(runtime, "load_library", lambda: lib)
    monkeypatch.setattr(runtime, "_torch", lambda: torch)
    monkeypatch.setattr(runtime, "_check_buffer", lambda *a: None)
    monkeypatch.setattr(runtime, "_raw_stream", lambda t: 5)
    return got


def _kernel():
    return lower_intent_to_hip_kernel(softmax_inner_ir(), shape_bindings={"M": 5, "N": 96})


def _buffers():
    import torch

    return {"input_ptr": torch.zeros(5, 96), "output_ptr": torch.zeros(5, 96)}


class _Slots:
    __slots__ = FIELDS

    def __init__(self, k):
        for f in FIELDS:
            setattr(self, f, getattr(k, f))


def _as(kind, k):
    values = {f: getattr(k, f) for f in FIELDS}
    return {"lowered": lambda: k, "slots": lambda: _Slots(k), "class": lambda: type("K", (), values),
            "tuple": lambda: namedtuple("K", FIELDS)(**values), "namespace": lambda: SimpleNamespace(**values)}[kind]()


@pytest.mark.parametrize("kind", ["lowered", "namespace", "slots", "tuple", "class"])
def test_any_object_with_the_fields_is_launched(calls, kind):
    lowered, b = _as(kind, _kernel()), _buffers()
    for _ in range(2):
        launch_lowered(lowered, b)
    assert len(calls) == 2 and calls[0] == calls[1]
    assert calls[0][:2] == (b["input_ptr"].data_ptr(), b["output_ptr"].data_ptr()) and calls[0][-1] == 5


class _Named:
    """Buffers with the two operations that a launch needs."""

    def __init__(self, d):
        self.d = d

    def __contains__(self, n):
        return n in self.d

    def __getitem__(self, n):
        return self.d[n]


def test_buffers_need_only_membership_and_lookup(calls):
    k, b = _kernel(), _buffers()
    launch_lowered(k, _Named(b))
    assert calls[0][:2] == (b["input_ptr"].data_ptr(), b["output_ptr"].data_ptr())
    del b["output_ptr"]
    with pytest.raises(runtime.HipRuntimeError, match="missing buffer for output_ptr"):
        launch_lowered(k, _Named(b))


def test_an_argument_outside_the_io_spec_is_passed(calls):
    """A call plan may name a tensor that io_spec does not describe: it is passed unchecked."""
    import torch

    k, b = _kernel(), _buffers()
    b["extra"] = torch.zeros(3)
    lowered = SimpleNamespace(io_spec=k.io_spec, bindings=k.bindings, kernel_id=k.kernel_id,
                              call_args=(*k.call_args, ("tensor", "extra")))
    launch_lowered(lowered, b)
    assert calls[0][-2] == b["extra"].data_ptr()


def test_call_args_changed_in_place_are_seen(calls):
    k, b = _kernel(), _buffers()
    for make in (list, lambda a: tuple(list(x) for x in a)):  # a list of pairs, a tuple of lists
        lowered = SimpleNamespace(io_spec=k.io_spec, bindings=k.bindings, kernel_id=k.kernel_id,
                                  call_args=make(k.call_args))
        launch_lowered(lowered, b)
        at = [i for i, (kind, _) in enumerate(lowered.call_args) if kind == "i64"][0]
        if isinstance(lowered.call_args, list):
            lowered.call_args[at] = ("i64", 3)
        else:
            lowered.call_args[at][1] = 3
        launch_lowered(lowered, b)
        assert calls[-2][at] == 5 and calls[-1][at] == 3


@pytest.mark.parametrize("dim", ["N", {"kind": "const", "value": 96}])
def test_io_spec_changed_in_place_is_seen(calls, dim):
    """A dtype, a dim in a shape, or something inside a dim that is neither a name nor a number."""
    plain = _kernel().io_spec["tensors"]["input_ptr"]
    tensors = {"input_ptr": {"dtype": "f32", "shape": [5, 96]}, "output_ptr": dict(plain)}
    spec = runtime._tensors_copy(tensors)
    assert spec == tensors
    tensors["input_ptr"]["shape"][1] = 97
    assert spec != tensors
    spec = runtime._tensors_copy(tensors)
    tensors["output_ptr"]["dtype"] = "f16"
    assert spec != tensors
    tensors["output_ptr"]["shape"] = [dim]
    spec = runtime._tensors_copy(tensors)
    if isinstance(dim, dict):
        dim["value"] = 7
        assert spec != tensors
