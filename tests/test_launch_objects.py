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
