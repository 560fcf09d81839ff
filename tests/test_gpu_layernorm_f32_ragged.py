"""f32 LayerNorm over rows that start at any 4-byte boundary (layernorm_f32.hip, kU): row lengths
at the edges of each register form, every tensor at an offset of its own, against the formula in
float64 on the host, and nothing written outside y.

Bounds: the sums of N f32 terms in a tree of at most 64 steps plus a wave's fold carry at most
~70 roundings of 2^-24 relative to the terms' magnitude; x is N(0, 1) + 1, so mean and variance are
of order one and 1e-5 covers them with a factor of two to spare, y (|y| <= ~6) likewise."""

import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

P = ctypes.c_void_p


@pytest.mark.parametrize("M,N", [(300001, 4), (270000, 7), (140001, 16), (70000, 33), (66003, 64), (40001, 101),
                                 (9001, 129), (8200, 255), (8193, 256)])
def test_layernorm_f32_many_short_rows(hip, M, N):
    """Two rows per lane group (grids of 1024 workgroups and more): every row against float64."""
    import torch

    g = torch.Generator(device="cuda")
    g.manual_seed(N)
    x = torch.randn((M, N), generator=g, device="cuda") + 1.0
    w, b = 1 + 0.1 * torch.randn(N, generator=g, device="cuda"), 0.1 * torch.randn(N, generator=g, device="cuda")
    y = torch.full((M * N + 16,), 7.0, device="cuda")
    mean, rstd = torch.empty(M, device="cuda"), torch.empty(M, device="cuda")
    print(f"[case] layernorm f32 short rows M={M} N={N}", flush=True)
    st = hip.ihip_layernorm_rows_f32(P(x.data_ptr()), P(w.data_ptr()), P(b.data_ptr()), P(y.data_ptr()),
                                     P(mean.data_ptr()), P(rstd.data_ptr()), M, N, ctypes.c_float(1e-5),
                                     P(torch.cuda.current_stream().cuda_stream))
    assert st == 0, hip.ihip_last_error().decode()
    xd = x.double()
    m = xd.mean(dim=1, keepdim=True)
    r = 1.0 / torch.sqrt(((xd - m) ** 2).mean(dim=1, keepdim=True) + 1e-5)
    # d = x - mean carries 2^-22 of |x| + |mean|, times rstd (short rows can be nearly constant)
    bound = 1e-5 + 1e-6 * (xd.abs() + m.abs() + 1) * r * (1 + (xd - m).abs() * r * r)
    assert (((y[:M * N].view(M, N).double() - ((xd - m) * r * w.double() + b.double())).abs()) <= bound).all()
    assert ((mean.double() - m[:, 0]).abs() <= 1e-6 * (1 + m[:, 0].abs())).all()
    assert ((rstd.double() - r[:, 0]).abs() <= 1e-5 * r[:, 0] * (1 + r[:, 0])).all()
    assert (y[M * N:] == 7.0).all()


@pytest.mark.parametrize("N", [1, 2, 3, 4, 5, 7, 255, 256, 257, 259, 511, 515, 1023, 1027, 2049, 2051, 4095, 4097, 4099,
                               4100, 4101, 8191, 8195, 16387, 32771, 65537, 65539, 65540])
@pytest.mark.parametrize("ox,ow,ob,oy", [(0, 0, 0, 0), (1, 2, 3, 0), (0, 1, 0, 3), (3, 0, 2, 1)])
def test_layernorm_f32_rows_at_any_4_byte_boundary(hip, N, ox, ow, ob, oy):
    import torch

    M = 9
    rng = np.random.default_rng(N * 64 + ox * 16 + oy)
    x = (rng.standard_normal((M, N)) + 1.0).astype(np.float32)
    w = (1 + 0.1 * rng.standard_normal(N)).astype(np.float32)
    b = (0.1 * rng.standard_normal(N)).astype(np.float32)

    def dev(a, off):
        buf = torch.full((a.size + off + 8,), 7.0, device="cuda")
        buf[off:off + a.size] = torch.from_numpy(a.ravel()).cuda()
        return buf, buf.data_ptr() + 4 * off

    (_x, px), (_w, pw), (_b, pb) = dev(x, ox), dev(w, ow), dev(b, ob)
    ybuf, py = dev(np.full((M, N), 7.0, np.float32), oy)
    mean, rstd = torch.empty(M, device="cuda"), torch.empty(M, device="cuda")
    print(f"[case] layernorm f32 N={N} offsets x{ox} w{ow} b{ob} y{oy}", flush=True)
    st = hip.ihip_layernorm_rows_f32(P(px), P(pw), P(pb), P(py), P(mean.data_ptr()), P(rstd.data_ptr()), M, N,
                                     ctypes.c_float(1e-5), P(torch.cuda.current_stream().cuda_stream))
    assert st == 0, hip.ihip_last_error().decode()
    torch.cuda.synchronize()
    xd = x.astype(np.float64)
    m = xd.mean(axis=1, keepdims=True)
    r = 1.0 / np.sqrt(((xd - m) ** 2).mean(axis=1, keepdims=True) + 1e-5)
    got = ybuf.cpu().numpy()
    # N = 1 has variance 0 and rstd 316: the mean is exact, so d = 0 and y = b
    np.testing.assert_allclose(got[oy:oy + M * N].reshape(M, N), (xd - m) * r * w + b, rtol=1e-5, atol=1e-5 * r.max())
    np.testing.assert_allclose(mean.cpu().numpy(), m[:, 0], rtol=1e-5, atol=1e-6)
    np.testing.assert_allclose(rstd.cpu().numpy(), r[:, 0], rtol=1e-5)
    assert (got[:oy] == 7.0).all() and (got[oy + M * N:] == 7.0).all(), "written outside y"
