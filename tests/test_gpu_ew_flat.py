"""The flat form of element-wise programs (ewjit.hip plan_flat): every operand form it accepts and
the ones it must leave to the row form, at row lengths around the run width, in every type, with
bases off their vectors' alignment.  The program only multiplies, adds, compares and selects, each
correctly rounded, so the native result must equal the interpreter kernel's bit for bit."""

import ctypes
import random

import pytest

from intent_ir_amd.ewprogram import OP, EwProgram
from intent_ir_amd.runtime import (EW_MODE_INTERP, EW_MODE_NATIVE, elementwise_source, ew_program_args, torch_dtype)

CODE = ((OP["load"], 0, 0, 0, 0, 0.0), (OP["load"], 1, 1, 0, 0, 0.0), (OP["load"], 2, 2, 0, 0, 0.0),
        (OP["mul"], 3, 0, 1, 0, 0.0), (OP["add"], 3, 3, 2, 0, 0.0), (OP["gt"], 4, 0, 2, 0, 0.0),
        (OP["where"], 5, 4, 3, 1, 0.0), (OP["store"], 0, 3, 0, 0, 0.0), (OP["store"], 0, 5, 1, 0, 0.0))

# (shape, flat): row lengths below, at and above the 4- and 8-element run, odd ones, ranks 1-4; flat
# says whether dense operands at aligned bases take the flat form (f32: 4 elements a run)
SHAPES = [((1,), False), ((3,), False), ((5,), True), ((4099,), True), ((7, 1), True), ((1000, 3), True), ((33, 4), True),
          ((257, 7), True), ((300, 8), True), ((129, 24), True), ((77, 257), True), ((5, 1021), True), ((9, 1024), False),
          ((64, 1000), False), ((3, 4, 65), True), ((2, 3, 5, 17), True), ((2, 1, 3, 1030), True), ((96,), False), ((1, 2280), False),
          ((2000, 280), True)]
KINDS = ("dense", "column", "row", "scalar")


def _strides(kind, sh):
    d0, d1, d2, d3 = sh
    return {"dense": (d1 * d2 * d3, d2 * d3, d3, 1), "column": (0, 0, 0, 1), "row": (d1 * d2, d2, 1, 0),
            "scalar": (0, 0, 0, 0), "outer": (1, 0, 0, 0)}[kind]


def _program(shape, kinds):
    sh = (1,) * (4 - len(shape)) + tuple(shape)
    return EwProgram(CODE, tuple((n, _strides(k, sh)) for n, k in zip("abc", kinds)), ("y", "z"), tuple(shape)), sh


@pytest.mark.parametrize("shape,flat", SHAPES)
def test_flat_form_is_taken_for_short_and_ragged_rows(shape, flat):
    """CPU: which source a launch compiles; inputs indexed along an outer axis only never go flat."""
    types = {n: "f32" for n in "abcyz"}
    ptrs = {n: 0x100000 * (i + 1) for i, n in enumerate("abcyz")}
    for kinds in (("dense", "dense", "dense"), ("dense", "column", "row"), ("scalar", "dense", "column")):
        assert ("ldf<0, 'u'>(a.in" in elementwise_source(_program(shape, kinds)[0], ptrs, types)) == flat
    if len(shape) == 4:
        src = elementwise_source(_program(shape, ("dense", "outer", "dense"))[0], ptrs, types)
        assert "ldf<0, 'u'>(a.in" not in src


@pytest.mark.parametrize("shape,flat", [((34161, 168), False), ((3416, 168), True), ((160006, 140), True), ((18000, 280), False),
                                        ((1500, 280), True), ((60000, 260), True), ((2017, 2280), False), ((300, 2280), True),
                                        ((3000, 1028), True), ((8000, 2280), True), ((8000, 2560), False)])
def test_flat_form_against_the_space_moved(shape, flat):
    """CPU: idle lanes count for less where the operands (4 bytes: one read and two written) move 16 MB or more."""
    types = {n: "f32" for n in "abcyz"}
    ptrs = {n: 0x100000 * (i + 1) for i, n in enumerate("abcyz")}
    prog = _program(shape, ("dense", "column", "row"))[0]
    assert ("ldf<0, 'u'>(a.in" in elementwise_source(prog, ptrs, types)) == flat


@pytest.mark.gpu
@pytest.mark.parametrize("types", [("f32", "f32", "f32", "f32", "bool"), ("bf16", "bf16", "bf16", "bf16", "f16"),
                                   ("f16", "bool", "bf16", "f16", "bool"), ("i32", "f32", "bool", "i32", "bf16")])
@pytest.mark.parametrize("shape", [s for s, _ in SHAPES])
def test_flat_form_equals_the_interpreter_kernel(hip, shape, types):
    import torch

    rng = random.Random(str((shape, types)))
    gen = torch.Generator(device="cuda")
    gen.manual_seed(len(shape) * 1000 + shape[-1])
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for trial in range(4):
        kinds = [rng.choice(KINDS) for _ in range(3)]
        prog, sh = _program(shape, kinds)
        total = sh[0] * sh[1] * sh[2] * sh[3]
        offs = [rng.choice((0, 0, 1, 3)) for _ in range(5)]
        dts = dict(zip("abcyz", types))
        size = {"dense": total, "column": sh[3], "row": sh[0] * sh[1] * sh[2], "scalar": 1}
        bufs = {}
        for n, k, off in zip("abc", kinds, offs):
            v = torch.randint(-40, 40, (size[k] + off,), generator=gen, device="cuda").float() / 8
            bufs[n] = (v > 0 if dts[n] == "bool" else v.to(torch_dtype(dts[n])))[off:]
        print(f"[case] flat {shape} {types} {kinds} offsets {offs}", flush=True)
        got = {}
        for mode in (EW_MODE_NATIVE, EW_MODE_INTERP):
            whole = {}
            for n, off in zip("yz", offs[3:]):  # 8 guard elements on either side of each output
                whole[n] = torch.ones(total + off + 16, device="cuda").to(torch_dtype(dts[n]))
                bufs[n] = whole[n][8 + off:8 + off + total]
            args = ew_program_args(prog, {n: t.data_ptr() for n, t in bufs.items()}, dts)
            keep = args.pop()
            prev = hip.ihip_elementwise_mode(mode)
            try:
                st = hip.ihip_elementwise_program(*args, stream)
            finally:
                hip.ihip_elementwise_mode(prev)
            assert st == 0, hip.ihip_last_error().decode()
            torch.cuda.synchronize()
            del keep
            got[mode] = whole
        for n in "yz":
            assert torch.equal(got[EW_MODE_NATIVE][n], got[EW_MODE_INTERP][n]), f"{n} differs"


@pytest.mark.gpu
@pytest.mark.parametrize("dt,V", [("f32", 4), ("bf16", 8), ("i32", 4)])
@pytest.mark.parametrize("total", [9, 64, 65, 67, 129, 257, 1025])  # in runs of V, and 1 or 3 elements more
def test_flat_form_in_place(hip, dt, V, total):
    """An output may be an input: the last run shares elements with one of another wave or workgroup."""
    import torch

    from intent_ir_amd import launch_lowered, lower_intent_to_hip_kernel

    N = total // 64 * 64 * V + total % 64
    ir = {"name": "bump", "tensors": {n: {"dtype": dt, "shape": ["M", "N"]} for n in "xyb"},
          "ops": [{"op": "add", "inputs": ["x", "b"], "output": "y"}], "outputs": ["y"]}
    k = lower_intent_to_hip_kernel(ir, shape_bindings={"M": 1, "N": N})
    x = torch.arange(N, device="cuda").remainder(50).to(torch_dtype(dt)).view(1, N)
    b = torch.ones_like(x)
    want = x + b
    print(f"[case] flat in place {dt} N={N}", flush=True)
    launch_lowered(k, {"x": x, "b": b, "y": x})
    torch.cuda.synchronize()
    assert torch.equal(x, want)
