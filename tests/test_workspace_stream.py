"""launch_lowered's workspace on an explicit stream: the block must come from that stream's pool.  A
block of the current stream's pool may have just been freed there while kernels queued on that
stream still use it, and nothing makes the launch's stream wait for them."""

import contextlib
from types import SimpleNamespace

import pytest

from intent_ir_amd import launch_lowered, lower_intent_to_hip_kernel
from intent_ir_amd import runtime
from intent_ir_amd.configs import matmul_bias_relu2d_ir

SHAPE = {"M": 64, "N": 192, "K": 8192}  # f32: K is cut into segments


@pytest.mark.parametrize("given", [False, True])
def test_workspace_is_allocated_on_the_launch_stream(monkeypatch, given):
    """CPU: which stream is current when the workspace is allocated, and what the entry point gets."""
    import torch

    k = lower_intent_to_hip_kernel(matmul_bias_relu2d_ir("f32"), shape_bindings=SHAPE)
    assert k.call_args[-1][0] == "workspace"
    current, at_alloc, passed = ["current"], [], []
    empty = torch.empty

    def fake_empty(*shape, device=None, **kw):
        at_alloc.append(current[-1])
        return empty(*shape, **kw)

    @contextlib.contextmanager
    def fake_stream(s):
        current.append(s)
        yield
        current.pop()

    monkeypatch.setattr(torch, "empty", fake_empty)
    monkeypatch.setattr(torch.cuda, "stream", fake_stream)
    monkeypatch.setattr(torch.Tensor, "record_stream", lambda self, s: None)
    monkeypatch.setattr(runtime, "_torch", lambda: torch)
    monkeypatch.setattr(runtime, "_check_buffer", lambda *a: None)
    monkeypatch.setattr(runtime, "_raw_stream", lambda t: 5)
    plan = runtime._call_plan(k)
    plan.fn = lambda *args: passed.append(args) or 0
    s = SimpleNamespace(cuda_stream=7)
    launch_lowered(k, {n: empty(1) for n in ("A", "B", "bias", "C")}, stream=s if given else None)
    assert at_alloc == [s if given else "current"]
    assert passed[0][-1] == (7 if given else 5) and passed[0][-3] != 0
    assert current == ["current"]


@pytest.mark.gpu
@pytest.mark.parametrize("ir", ["f32", "bf16"])
def test_split_product_on_another_stream_after_a_free(hip, ir):
    """Blocks of the workspace's size are freed on the current stream with fills still queued there."""
    import torch

    b = SHAPE if ir == "f32" else {"M": 16, "N": 1024, "K": 8192}
    k = lower_intent_to_hip_kernel(matmul_bias_relu2d_ir(ir), shape_bindings=b)
    nbytes = k.call_args[-1][1]
    assert k.call_args[-1][0] == "workspace" and nbytes > 0
    dt = {"f32": torch.float32, "bf16": torch.bfloat16}[ir]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(3)

    def ints(*shape):  # every sum is exact whatever its order
        return torch.randint(-3, 4, shape, generator=gen, device="cuda").float()

    A, B, bias = ints(b["M"], b["K"]), ints(b["K"], b["N"]), ints(b["N"])
    want = torch.relu(A.double() @ B.double() + bias.double()).to(dt)
    bufs = {"A": A.to(dt), "B": B.to(dt), "bias": bias}
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    for i in range(8):
        print(f"[case] {ir} product on another stream, pass {i}", flush=True)
        C = torch.zeros(b["M"], b["N"], dtype=dt, device="cuda")
        torch.cuda.synchronize()
        junk = [torch.empty(nbytes, dtype=torch.uint8, device="cuda") for _ in range(4)]
        for _ in range(20):
            for j in junk:
                j.fill_(0xFF)
        del junk, j
        launch_lowered(k, {**bufs, "C": C}, stream=s)
        torch.cuda.synchronize()
        assert torch.equal(C, want)
