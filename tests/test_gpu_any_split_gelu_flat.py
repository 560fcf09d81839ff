"""reduce_any over few long rows (rows.hip reduce_any_rows_split) and the bf16 GELU chain over rows
off 16-byte alignment (elementwise.hip bias_gelu_axpy_bf16_flat): edges of their segments and runs."""

import ctypes

import numpy as np
import pytest

from intent_ir_amd.dtypes import bf16_bits_to_f32, f32_to_bf16_bits

pytestmark = pytest.mark.gpu
P = ctypes.c_void_p


def _stream(torch):
    return P(torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize("M,N", [(1, 16384), (3, 16389), (2, 70003), (255, 16387), (511, 16384), (5, 1048583)])
@pytest.mark.parametrize("off", [0, 1, 3])
def test_any_split_finds_one_element_anywhere(hip, M, N, off):
    """One element that differs per row (or none), at the ends of the row, of its aligned body and of
    its segments, against c = 0 (with -0.0 elsewhere) and c = 1; out holds garbage before the call."""
    import torch

    spots = [None, 0, 1, 3, 4, N // 2, 4096 * 4 - 1, min(N - 1, 4096 * 4 + 3), N - 5, N - 2, N - 1]
    for c in (0.0, 1.0):
        for first in range(0, len(spots), max(1, min(M, len(spots)))):
            buf = torch.full((M * N + off,), -0.0 if c == 0.0 else 1.0, device="cuda")
            x = buf[off:].view(M, N)
            want = np.zeros(M, bool)
            for r in range(M):
                s = spots[(first + r) % len(spots)]
                if s is not None:
                    x[r, s] = float("nan") if r % 3 == 0 else 1e-45 if c == 0.0 else 2.0
                    want[r] = True
            out = torch.full((M + 8,), 7, dtype=torch.uint8, device="cuda")
            print(f"[case] any split M={M} N={N} off={off} c={c} from spot {first}", flush=True)
            st = hip.ihip_reduce_any_rows_f32(P(buf.data_ptr() + 4 * off), P(out.data_ptr()), M, N, ctypes.c_float(c),
                                              _stream(torch))
            assert st == 0, hip.ihip_last_error().decode()
            torch.cuda.synchronize()
            h = out.cpu().numpy()
            np.testing.assert_array_equal(h[:M], want)
            assert (h[M:] == 7).all()


@pytest.mark.parametrize("M,N", [(1, 65536), (3, 65551), (400, 70001)])
@pytest.mark.parametrize("off", [0, 5, 15])
def test_any_split_over_bytes(hip, M, N, off):
    import torch

    buf = torch.zeros(M * N + off, dtype=torch.uint8, device="cuda")
    x = buf[off:].view(M, N)
    spots = [None, 0, 15, 16, N // 2, 16 * 1024 - 1, 16 * 1024, N - 17, N - 1]
    want = np.zeros(M, bool)
    for r in range(M):
        s = spots[(r + off) % len(spots)]
        if s is not None:
            x[r, s] = 1
            want[r] = True
    out = torch.full((M + 8,), 7, dtype=torch.uint8, device="cuda")
    print(f"[case] any split u8 M={M} N={N} off={off}", flush=True)
    st = hip.ihip_reduce_any_rows_u8(P(buf.data_ptr() + off), P(out.data_ptr()), M, N, _stream(torch))
    assert st == 0, hip.ihip_last_error().decode()
    torch.cuda.synchronize()
    h = out.cpu().numpy()
    np.testing.assert_array_equal(h[:M], want)
    assert (h[M:] == 7).all()


@pytest.mark.parametrize("M,N", [(1, 8), (1, 9), (3, 9), (5, 15), (700, 8), (301, 17), (40, 257), (9, 1603), (3, 4099),
                                 (2000, 23), (233017, 9), (123362, 17), (1309, 1603), (1, 2097167)])
@pytest.mark.parametrize("ox,ob,oy", [(0, 0, 0), (1, 0, 0), (3, 5, 7), (0, 1, 4)])
@pytest.mark.parametrize("alpha", [0.5, 0.0])
def test_gelu_rows_at_any_2_byte_boundary(hip, M, N, ox, ob, oy, alpha):
    """Against the formula in float64: half a unit of bf16 (8 significant bits: 2^-8 relative) and the kernel's f32
    arithmetic (some 2^-20 of |z| + |x|)."""
    import torch

    rng = np.random.default_rng(M * 131 + N)
    x = f32_to_bf16_bits(rng.standard_normal((M, N)).astype(np.float32) * 2)
    b = f32_to_bf16_bits(rng.standard_normal(N).astype(np.float32))

    def dev(a, off):
        t = torch.full((a.size + off + 8,), 0x1234, dtype=torch.int16, device="cuda")
        t[off:off + a.size] = torch.from_numpy(a.reshape(-1).view(np.int16)).cuda()
        return t

    xd, bd, yd = dev(x, ox), dev(b, ob), dev(np.zeros(M * N, np.uint16), oy)
    print(f"[case] gelu flat M={M} N={N} offsets {ox} {ob} {oy} alpha={alpha}", flush=True)
    st = hip.ihip_bias_gelu_tanh_axpy_bf16(P(xd.data_ptr() + 2 * ox), P(bd.data_ptr() + 2 * ob), P(yd.data_ptr() + 2 * oy),
                                           M, N, ctypes.c_float(alpha), _stream(torch))
    assert st == 0, hip.ihip_last_error().decode()
    torch.cuda.synchronize()
    h = yd.cpu().numpy().view(np.uint16)
    xf, bf = bf16_bits_to_f32(x).astype(np.float64), bf16_bits_to_f32(b).astype(np.float64)
    z = xf + bf
    ref = alpha * z * 0.5 * (1 + np.tanh(np.sqrt(2 / np.pi) * (z + 0.044715 * z ** 3))) + xf
    got = bf16_bits_to_f32(h[oy:oy + M * N].reshape(M, N)).astype(np.float64)
    assert (np.abs(got - ref) <= 2.0 ** -8 * np.abs(ref) + 2.0 ** -19 * (np.abs(z) + np.abs(xf))).all()
    assert (h[:oy] == 0x1234).all() and (h[oy + M * N:] == 0x1234).all(), "written outside y"


@pytest.mark.parametrize("M,N", [(1, 9), (1, 513), (3, 171), (1, 2049), (1, 8193), (7, 1171), (5, 1639), (683, 771),
                                 (1, 2097161), (233019, 9), (1031, 2049), (2049, 1025)])
def test_gelu_in_place(hip, M, N):
    """y may be x: the runs at the end, which share elements across waves and workgroups, included."""
    import torch

    gen = torch.Generator(device="cuda")
    gen.manual_seed(M * N)
    x = torch.randn(M, N, device="cuda", generator=gen).bfloat16()
    b = torch.randn(N, device="cuda", generator=gen).bfloat16()
    y = torch.empty_like(x)
    print(f"[case] gelu in place M={M} N={N}", flush=True)
    for out in (y, x):
        st = hip.ihip_bias_gelu_tanh_axpy_bf16(P(x.data_ptr()), P(b.data_ptr()), P(out.data_ptr()), M, N,
                                               ctypes.c_float(0.5), _stream(torch))
        assert st == 0, hip.ihip_last_error().decode()
    torch.cuda.synchronize()
    assert torch.equal(x, y)
