"""launch_lowered's plan (runtime._CallPlan) holds nothing of a buffer: every call's own buffers are
checked and used, from several threads and streams, and the lowered kernel still copies and pickles."""

import copy
import pickle
import threading

import pytest

from intent_ir_amd import HipRuntimeError, launch_lowered, lower_intent_to_hip_kernel
from intent_ir_amd.configs import WORKLOADS, softmax_inner_ir

pytestmark = pytest.mark.gpu


def _chain(M, N):
    def t(*shape):
        return {"dtype": "f32", "shape": list(shape)}

    ir = {"name": "scale_add", "tensors": {"x": t("M", "N"), "b": t("N"), "u": t("M", "N"), "y": t("M", "N")},
          "ops": [{"op": "mul", "inputs": ["x"], "output": "u", "attrs": {"mul_factor": 2.0}},
                  {"op": "add", "inputs": ["u", "b"], "output": "y"}], "outputs": ["y"]}
    return lower_intent_to_hip_kernel(ir, shape_bindings={"M": M, "N": N})


def test_every_call_checks_and_uses_its_own_buffers(hip):
    import torch

    M, N = 5, 96
    k = lower_intent_to_hip_kernel(softmax_inner_ir(), shape_bindings={"M": M, "N": N})
    for i in range(3):
        x = torch.randn(M, N, device="cuda")
        y = torch.full((M, N), 7.0, device="cuda")
        launch_lowered(k, {"input_ptr": x, "output_ptr": y})
        torch.testing.assert_close(y, torch.softmax(x, dim=1))
    y2 = torch.empty(M * N, device="cuda")  # the same number of elements in another shape is accepted
    launch_lowered(k, {"input_ptr": x, "output_ptr": y2})
    assert torch.equal(y2.view(M, N), y)
    good = {"input_ptr": x, "output_ptr": y}
    for name, bad, why in (("input_ptr", x.half(), "dtype"), ("input_ptr", x[:, ::2], "shape"),
                           ("input_ptr", torch.randn(N, M, device="cuda").t(), "contiguous"),
                           ("output_ptr", torch.empty(M, N), "not a ROCm device"), ("input_ptr", None, "torch tensor"),
                           ("output_ptr", torch.empty(M + 1, N, device="cuda"), "shape")):
        with pytest.raises(HipRuntimeError, match=why):
            launch_lowered(k, {**good, name: bad})
    with pytest.raises(HipRuntimeError, match="missing buffer for output_ptr"):
        launch_lowered(k, {"input_ptr": x})


@pytest.mark.parametrize("make", [lambda: _chain(64, 100),
                                  lambda: lower_intent_to_hip_kernel(WORKLOADS["matmul"].ir(),
                                                                     shape_bindings={"M": 16, "N": 1024, "K": 4096})],
                         ids=["program", "workspace"])
def test_copies_and_pickles_after_a_launch(hip, make):
    import torch

    k = make()
    bufs = {n: torch.randn([k.bindings.get(d, d) for d in s["shape"]], device="cuda").to(
        {"f32": torch.float32, "bf16": torch.bfloat16}[s["dtype"]]) for n, s in k.io_spec["tensors"].items()}
    launch_lowered(k, bufs)
    out = bufs[k.output_names[0]].clone()
    for other in (copy.copy(k), copy.deepcopy(k), pickle.loads(pickle.dumps(k))):
        assert other == k
        bufs[k.output_names[0]].zero_()
        launch_lowered(other, bufs)
        assert torch.equal(bufs[k.output_names[0]], out)


def test_one_kernel_from_several_threads_and_streams(hip):
    """Threads share the plan and its program tables' templates; each call fills tables of its own."""
    import torch

    M, N, threads, rounds = 300, 1000, 4, 40
    k = _chain(M, N)
    data = [[(torch.randn(M, N, device="cuda"), torch.randn(N, device="cuda"), torch.empty(M, N, device="cuda"))
             for _ in range(rounds)] for _ in range(threads)]
    torch.cuda.synchronize()
    errors = []

    def work(i):
        try:
            s = torch.cuda.Stream()
            for x, b, y in data[i]:
                if i % 2:
                    launch_lowered(k, {"x": x, "b": b, "y": y}, stream=s)
                else:
                    with torch.cuda.stream(s):
                        launch_lowered(k, {"x": x, "b": b, "y": y})
            s.synchronize()
        except Exception as e:  # noqa: BLE001 - reported below
            errors.append(e)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(threads)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors
    for rows in data:
        for x, b, y in rows:
            assert torch.equal(y, x * 2.0 + b)


def test_a_changed_io_spec_is_seen(hip):
    import torch

    k = lower_intent_to_hip_kernel(softmax_inner_ir(), shape_bindings={"M": 5, "N": 96})
    good = {"input_ptr": torch.randn(5, 96, device="cuda"), "output_ptr": torch.empty(5, 96, device="cuda")}
    launch_lowered(k, good)
    k.io_spec["tensors"]["input_ptr"]["dtype"] = "f16"
    with pytest.raises(HipRuntimeError, match="dtype"):
        launch_lowered(k, good)
