"""The f32 product cut along K (gemm_f32.hip f32_split_plan, gemm_f32_reduce): integer operands, so
every order of the sums is exact and C must be too, at the edges of tiles, segments and layouts;
without a workspace the unsplit kernel runs, and gives the same."""

import ctypes

import numpy as np
import pytest

from intent_ir_amd.lowering import gemm_f32_split_plan

P = ctypes.c_void_p
SHAPES = [(46, 704, 8512), (1, 512, 1024), (64, 64, 256), (65, 63, 2051), (300, 300, 600), (130, 257, 1000), (7, 5, 4100),
          (1000, 129, 777), (512, 512, 512)]


@pytest.mark.parametrize("M,N,K", SHAPES + [(28, 80, 240), (6081, 271, 2560), (1000, 1001, 4096), (4096, 4096, 64),
                                            (1, 1, 100000), (3, 0, 64), (0, 5, 64)])
def test_lowering_follows_the_library(M, N, K):
    """CPU: the segments' workspace is the library's."""
    from intent_ir_amd.runtime import load_library

    S = gemm_f32_split_plan(M, N, K)[0]
    want = S * M * (-(-N // 4) * 4) * 4 if S > 1 else 0
    assert load_library().ihip_gemm_f32_workspace_size(M, N, K) == want


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("ta,tb", [(False, False), (False, True), (True, False), (True, True)])
def test_split_f32_product_is_exact_on_integers(hip, M, N, K, ta, tb):
    import torch

    S = gemm_f32_split_plan(M, N, K)[0]
    assert S > 1
    rng = np.random.default_rng(M + 3 * N + 7 * K)
    A = rng.integers(-4, 5, size=(K, M) if ta else (M, K)).astype(np.float32)
    B = rng.integers(-4, 5, size=(N, K) if tb else (K, N)).astype(np.float32)
    bias = rng.integers(-8, 9, size=N).astype(np.float32)
    a64, b64 = torch.from_numpy(A).cuda().double(), torch.from_numpy(B).cuda().double()
    full = ((a64.t() if ta else a64).contiguous() @ (b64.t() if tb else b64).contiguous()).cpu().numpy()
    need = hip.ihip_gemm_f32_workspace_size(M, N, K)
    for relu, bs, off in ((True, bias, 0), (False, None, 1)):
        def dev(x, pad):
            t = torch.zeros(x.size + pad, device="cuda")
            t[pad:] = torch.from_numpy(x.ravel()).cuda()
            return t

        a, b = dev(A, off), dev(B, 2 * off)
        bd = None if bs is None else torch.from_numpy(bs).cuda()
        want = full if bs is None else full + bs
        want = np.maximum(want, 0) if relu else want
        for ws_bytes in (need, need - 1, 0):
            c = torch.full((M * N + 16 + off,), 7.0, device="cuda")
            ws = torch.full((max(1, ws_bytes),), 0xFF, dtype=torch.uint8, device="cuda")  # NaN where nothing is written
            print(f"[case] f32 split M={M} N={N} K={K} ta={ta} tb={tb} S={S} off={off} ws={ws_bytes}", flush=True)
            st = hip.ihip_gemm_f32_bias_relu_ws(
                P(a.data_ptr() + 4 * off), P(b.data_ptr() + 8 * off), P(None if bd is None else bd.data_ptr()),
                P(c.data_ptr() + 4 * (8 + off)), M, N, K, int(ta), int(tb), int(relu), 0,
                P(ws.data_ptr() if ws_bytes else None), ws_bytes, P(torch.cuda.current_stream().cuda_stream))
            assert st == 0, hip.ihip_last_error().decode()
            torch.cuda.synchronize()
            h = c.cpu().numpy()
            lo = 8 + off
            np.testing.assert_array_equal(h[lo:lo + M * N].reshape(M, N), want.astype(np.float32))
            assert (h[:lo] == 7.0).all() and (h[lo + M * N:] == 7.0).all(), "written outside C"
