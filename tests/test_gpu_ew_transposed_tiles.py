"""Tiles of element-wise programs with inputs read across their unit-stride axis (ewjit.hip
plan_jit): 128 x 32 where every operand is 4 bytes wide, the staged ones are read in vectors and a
tile's output lines are its own (rows of at most 32 elements, or whole lines of a large space),
64 x 64 otherwise, at extents around both tiles, with aligned and unaligned bases.  The program only
adds and multiplies, each correctly rounded, so the native result must equal the interpreter
kernel's bit for bit."""

import ctypes

import pytest

from intent_ir_amd.ewprogram import OP, EwProgram
from intent_ir_amd.runtime import (EW_MODE_INTERP, EW_MODE_NATIVE, elementwise_source, ew_program_args, torch_dtype)

CODE = ((OP["load"], 0, 0, 0, 0, 0.0), (OP["load"], 1, 1, 0, 0, 0.0), (OP["load"], 2, 2, 0, 0, 0.0),
        (OP["mul"], 3, 0, 1, 0, 0.0), (OP["add"], 3, 3, 2, 0, 0.0), (OP["store"], 0, 3, 0, 0, 0.0))

# (batch, axis 2, axis 3), wide in f32
SHAPES = [((1, 128, 32), True), ((1, 127, 31), False), ((1, 65, 32), False), ((1, 68, 32), True), ((1, 64, 32), False),
          ((1, 129, 33), False), ((1, 128, 64), False), ((1, 130, 96), False), ((1, 200, 100), False),
          ((1, 520, 256), False), ((2, 256, 128), False), ((3, 100, 7), True), ((1, 1000, 1), False), ((1, 2, 1000), False),
          ((1, 1024, 1028), False), ((2, 255, 257), False), ((1, 1000, 20), True), ((5, 132, 31), True)]
# the same above 256 MB: whole lines only, and no more tiles of 128 x 32 than of 64 x 64
LARGE = [((1, 8192, 8192), True), ((1, 8192, 4128), True), ((1, 8192, 4100), False), ((1, 8192, 4112), False),
         ((1, 8191, 4128), False), ((1, 5800, 5888), False), ((1, 1048576, 33), False), ((1, 1048576, 32), True)]
TYPES = [("f32", "f32", "f32", "f32"), ("i32", "f32", "f32", "f32"), ("bf16", "f32", "f32", "f32"),
         ("f32", "f32", "f32", "f16"), ("f16", "f16", "f16", "f16")]


def _program(shape):
    b, r, c = shape
    return EwProgram(CODE, (("a", (r * c, 0, 1, r)), ("b", (r * c, 0, c, 1)), ("c", (0, 0, 0, 1))), ("y",), (b, 1, r, c))


@pytest.mark.parametrize("shape,wide", SHAPES + LARGE)
def test_tile_extents_follow_types_and_shape(shape, wide):
    """CPU: which tile a launch compiles, and the staging loads (ordinary for short rows up to 256 MB
    moved)."""
    ptrs = {n: 0x100000 * (i + 1) for i, n in enumerate("abcy")}
    for types in TYPES:
        src = elementwise_source(_program(shape), ptrs, dict(zip("abcy", types)))
        took = wide and all(t in ("f32", "i32") for t in types)
        assert ("#define EW_T2 128" in src) == took
        small = 8 * shape[0] * shape[1] * shape[2] <= 256e6
        assert ("ld4c<0>(p" in src or "ld4c<4>(p" in src) == (took and small)


@pytest.mark.parametrize("shape,ordinary", [((1, 86872, 143), True), ((1, 42668, 296), True), ((1, 108024, 76), True),
                                            ((1, 86873, 143), False), ((1, 40000, 143), False), ((1, 4096, 4100), False),
                                            ((1, 60000, 96), False), ((1, 117052, 128), True), ((1, 98304, 256), False),
                                            ((1, 100000, 143), False), ((2, 43436, 143), True)])
def test_staging_loads_of_64_x_64_tiles(shape, ordinary):
    """CPU: ordinary loads where they cost rotating buffers nothing; 4-byte operands only."""
    ptrs = {n: 0x100000 * (i + 1) for i, n in enumerate("abcy")}
    for types in TYPES[:3]:
        src = elementwise_source(_program(shape), ptrs, dict(zip("abcy", types)))
        assert "#define EW_T2 64" in src
        assert ("ld4c<" in src.split("ihip_ew_jit")[1]) == (ordinary and types[0] != "bf16")


@pytest.mark.parametrize("shape,wide", LARGE)
def test_wide_tiles_need_output_lines_of_their_own(shape, wide):
    """CPU: an output off a 128-byte boundary shares its lines between tiles; short rows do not mind."""
    ptrs = {n: 0x100000 * (i + 1) for i, n in enumerate("abcy")}
    ptrs["y"] += 16
    src = elementwise_source(_program(shape), ptrs, dict(zip("abcy", TYPES[0])))
    assert ("#define EW_T2 128" in src) == (wide and shape[2] <= 32)


@pytest.mark.gpu
@pytest.mark.parametrize("types", TYPES)
@pytest.mark.parametrize("shape", [s for s, _ in SHAPES] + [(1, 5800, 5888), (1, 8192, 4128), (1, 1048576, 32),
                                                             (1, 60000, 143), (1, 42668, 296)])
def test_tiled_form_equals_the_interpreter_kernel(hip, shape, types):
    import torch

    gen = torch.Generator(device="cuda")
    gen.manual_seed(shape[1] * 1000 + shape[2])
    prog, total = _program(shape), shape[0] * shape[1] * shape[2]
    dts = dict(zip("abcy", types))
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for off in (0, 1):
        print(f"[case] tiles {shape} {types} offset {off}", flush=True)
        bufs = {}
        for n in "abc":
            v = torch.randint(-40, 40, ((shape[2] if n == "c" else total) + off,), generator=gen, device="cuda") / 8
            bufs[n] = v.to(torch_dtype(dts[n]))[off:]
        got = {}
        for mode in (EW_MODE_NATIVE, EW_MODE_INTERP):
            whole = torch.ones(total + off + 16, device="cuda").to(torch_dtype(dts["y"]))  # guards around y
            bufs["y"] = whole[8 + off:8 + off + total]
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
        assert torch.equal(got[EW_MODE_NATIVE], got[EW_MODE_INTERP])
