"""The bf16 product with one small side (gemm_direct.hip): edges of its blocks, slabs and segments.

Operands are small integers, so every f32 sum is exact whatever its order, and C must equal the
exact product rounded to bf16, bit for bit, with and without the workspace its segments ask for."""

import ctypes

import numpy as np
import pytest

from intent_ir_amd.dtypes import f32_to_bf16_bits
from intent_ir_amd.lowering import _gemm_split_bytes as gemm_split_bytes
from intent_ir_amd.lowering import (gemm_direct_plan, gemm_direct_takes, gemm_pack_bytes, gemm_split_plan,
                                    gemm_workspace_bytes)

P = ctypes.c_void_p
GUARD = 64

# M at the row-fragment edges, N at the column-block edges and the 32/64/128-column blocks, K at the
# slab edges (whole slabs, a tail of 1 to 63, fewer slabs than waves), several segments
SHAPES = [(1, 16, 129), (15, 17, 191), (16, 63, 136), (17, 65, 193), (31, 64, 192), (32, 130, 200), (33, 66, 520),
          (64, 127, 1000), (65, 129, 327), (127, 71, 511), (128, 515, 263), (1, 1001, 2049), (7, 4097, 2056),
          (16, 1024, 8192), (48, 1000, 4104), (64, 300, 8191), (3, 16384, 136), (5, 28672, 2048), (20, 25601, 2100),
          (2, 8200, 2304), (32, 33000, 160), (17, 64, 512), (64, 512, 384), (65, 129, 771), (127, 71, 1023), (48, 392, 520)]


@pytest.mark.parametrize("M,N,K", SHAPES + [(64, 49152, 4096), (128, 65536, 999), (128, 263, 128), (16, 50256, 4096)])
@pytest.mark.parametrize("tb", [False, True])
def test_lowering_follows_the_library(M, N, K, tb):
    """CPU: the plan's workspace is the library's (ihip_gemm_workspace_size)."""
    from intent_ir_amd.runtime import load_library

    assert load_library().ihip_gemm_workspace_size(M, N, K, 0, int(tb)) == gemm_workspace_bytes(M, N, K, False, tb)


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("tb", [False, True])
def test_workspace_size_holds_what_a_fixed_tile_needs(M, N, K, tb):
    """CPU: the size has no tile argument, so it also covers tile = 128 or 256: the packed copies of
    ragged operands and the tiled kernel's partials, beside the few-row kernel's."""
    from intent_ir_amd.runtime import load_library

    size = load_library().ihip_gemm_workspace_size(M, N, K, 0, int(tb))
    tiled = gemm_pack_bytes(M, N, K, False, tb) + gemm_split_bytes(M, N, gemm_split_plan(M, N, -(-K // 8) * 8)[0])
    few = gemm_split_bytes(M, N, gemm_direct_plan(M, N, K, tb)[2]) if gemm_direct_takes(M, N, K, False, tb) else 0
    assert size == max(tiled, few)


def _run(hip, torch, A, B, bias, M, N, K, tb, relu, offs, ws_bytes):
    def dev(x, off):
        t = torch.zeros(x.size + off, dtype=torch.int16, device="cuda")
        t[off:] = torch.from_numpy(x.reshape(-1).view(np.int16)).cuda()
        return t

    a, b = dev(A, offs[0]), dev(B, offs[1])
    bd = None if bias is None else torch.from_numpy(bias).cuda()
    c = torch.full((M * N + 2 * GUARD + offs[2],), 0x1234, dtype=torch.int16, device="cuda")
    ws = torch.full((max(1, ws_bytes),), 0xFF, dtype=torch.uint8, device="cuda")  # NaN where nothing is written
    st = hip.ihip_gemm_bf16_bias_relu_ws(
        P(a.data_ptr() + 2 * offs[0]), P(b.data_ptr() + 2 * offs[1]), P(None if bd is None else bd.data_ptr()),
        P(c.data_ptr() + 2 * (GUARD + offs[2])), M, N, K, 0, int(tb), int(relu), 0, P(ws.data_ptr() if ws_bytes else None),
        ws_bytes, P(torch.cuda.current_stream().cuda_stream))
    assert st == 0, hip.ihip_last_error().decode()
    torch.cuda.synchronize()
    h = c.cpu().numpy().view(np.uint16)
    lo = GUARD + offs[2]
    assert (h[:lo] == 0x1234).all() and (h[lo + M * N:] == 0x1234).all(), "written outside C"
    return h[lo:lo + M * N].reshape(M, N)


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("tb", [False, True])
def test_direct_product_is_exact_on_integers(hip, M, N, K, tb):
    import torch

    if not gemm_direct_takes(M, N, K, False, tb):
        pytest.skip("this layout of the shape runs on the tiled kernels")
    rng = np.random.default_rng(M * 31 + N * 7 + K)
    Af = rng.integers(-4, 5, size=(M, K)).astype(np.float32)
    Bf = rng.integers(-4, 5, size=(K, N)).astype(np.float32)
    bias = rng.integers(-8, 9, size=N).astype(np.float32)
    full = (torch.from_numpy(Af).cuda().double() @ torch.from_numpy(Bf).cuda().double()).cpu().numpy()
    A, B = f32_to_bf16_bits(Af), f32_to_bf16_bits(np.ascontiguousarray(Bf.T) if tb else Bf)
    S = gemm_direct_plan(M, N, K, tb)[2]
    need = gemm_split_bytes(M, N, S)
    assert (need > 0) == (S > 1)
    for relu, bs, offs in ((True, bias, (0, 0, 0)), (False, None, (1, 3, 1)), (True, bias, (0, 1, 5))):
        ref = full if bs is None else full + bs
        want = f32_to_bf16_bits((np.maximum(ref, 0) if relu else ref).astype(np.float32))
        for ws in {0, need}:
            print(f"[case] direct M={M} N={N} K={K} tb={tb} S={S if ws else 1} offsets {offs}", flush=True)
            got = _run(hip, torch, A, B, bs, M, N, K, tb, relu, offs, ws)
            bad = (got != want) & ~((got == 0x8000) & (want == 0))  # a zero sum's sign is not at stake
            assert not bad.any(), f"{int(bad.sum())} elements differ, first at {np.argwhere(bad)[0]}"


@pytest.mark.gpu
@pytest.mark.parametrize("tb", [False, True])
def test_direct_product_keeps_nan_and_inf_to_their_rows_and_columns(hip, tb):
    """Rows and columns that are clamped reads, and k past K, must not leak a NaN or an inf."""
    import torch

    M, N, K = 19, 1003, 333
    rng = np.random.default_rng(5)
    Af, Bf = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((K, N)).astype(np.float32)
    Af[M - 1, K - 1] = np.nan   # the last row, read again by the lanes past it
    Bf[K - 1, N - 1] = np.inf   # the last column and k
    Bf[3, 5] = -np.inf
    A, B = f32_to_bf16_bits(Af), f32_to_bf16_bits(np.ascontiguousarray(Bf.T) if tb else Bf)
    print(f"[case] direct special operands tb={tb}", flush=True)
    got = _run(hip, torch, A, B, None, M, N, K, tb, False, (0, 0, 0), gemm_workspace_bytes(M, N, K, False, tb))
    f = (got.astype(np.uint32) << 16).view(np.float32)
    finite = np.ones((M, N), bool)
    finite[M - 1] = False
    finite[:, N - 1] = finite[:, 5] = False
    np.testing.assert_array_equal(np.isfinite(f), finite)
    assert np.isnan(f[M - 1]).all() and np.isinf(f[:M - 1, 5]).all()


def test_lowered_few_row_products_call_the_workspace_entry():
    """CPU: the entries without a workspace sum K in one chain, so the few-row kernel is the workspace
    entry's, with or without segments."""
    from intent_ir_amd import lower_intent_to_hip_kernel
    from intent_ir_amd.configs import matmul_bias_relu2d_ir

    for M, N, K, S in ((32, 32000, 4096, 1), (16, 1024, 8192, 16)):
        assert gemm_direct_takes(M, N, K, False, False) and gemm_direct_plan(M, N, K, False)[2] == S
        k = lower_intent_to_hip_kernel(matmul_bias_relu2d_ir(), shape_bindings={"M": M, "N": N, "K": K})
        assert k.kernel_id == "ihip_gemm_bf16_bias_relu_ws"
        assert k.call_args[-2:] == ((("null", None), ("i64", 0)) if S == 1 else
                                    (("i32", 0), ("workspace", gemm_split_bytes(M, N, S))))


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(16, 1024, 8192), (1, 264, 1000), (33, 520, 1003), (128, 513, 4096)])
def test_entries_without_a_workspace_give_the_same_bits_for_every_tile_and_layout(hip, M, N, K):
    """Also on shapes of the few-row kernel: one chain over K.  That kernel's result (the workspace
    entry, automatic tile) differs by the order of its f32 sums only: the two C are within their
    bf16 roundings (2^-8 of the value each) and their sums' bounds (K 2^-24 sum |a b| each)."""
    import torch

    assert gemm_direct_takes(M, N, K, False, False)
    rng = np.random.default_rng(M + N + K)
    Af, Bf = rng.standard_normal((M, K)).astype(np.float32), rng.standard_normal((K, N)).astype(np.float32)
    bias = torch.from_numpy(rng.standard_normal(N).astype(np.float32)).cuda()
    stream = P(torch.cuda.current_stream().cuda_stream)

    def dev(x):
        return torch.from_numpy(f32_to_bf16_bits(np.ascontiguousarray(x)).view(np.int16)).cuda().view(torch.bfloat16)

    op = {("A", False): dev(Af), ("A", True): dev(Af.T), ("B", False): dev(Bf), ("B", True): dev(Bf.T)}

    def run(name, ta, tb, *tail):
        c = torch.full((M, N), float("nan"), dtype=torch.bfloat16, device="cuda")
        flags = () if name.endswith("relu") else (int(ta), int(tb))
        st = getattr(hip, name)(P(op["A", ta].data_ptr()), P(op["B", tb].data_ptr()), P(bias.data_ptr()), P(c.data_ptr()),
                                M, N, K, *flags, 0, *tail, stream)
        assert st == 0, hip.ihip_last_error().decode()
        torch.cuda.synchronize()
        return c

    print(f"[case] entries without a workspace {M}x{N}x{K}", flush=True)
    want = run("ihip_gemm_bf16_bias_relu", False, False)
    for ta in (False, True):
        for tb in (False, True):
            assert torch.equal(run("ihip_gemm_bf16_bias_relu_t", ta, tb), want), (ta, tb)
            for tile in (0, 128, 256):
                assert torch.equal(run("ihip_gemm_bf16_bias_relu_ex", ta, tb, tile), want), (ta, tb, tile)
    mag = op["A", False].double().abs() @ op["B", False].double().abs()
    for tb in (False, True):
        got = run("ihip_gemm_bf16_bias_relu_ws", False, tb, 0, P(None), 0)
        err = (got.double() - want.double()).abs()
        assert (err <= want.double().abs() * 2.0 ** -7 + 2 * K * 2.0 ** -24 * mag).all()
