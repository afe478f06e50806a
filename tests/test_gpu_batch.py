"""The batch kernel (bw_qlinear_ws from 5, 17 or so rows up to 2048) against the oracle: every format, row counts at the edges of
its row tiles, columns and K that end inside tiles and rounds, K cut across workgroups or not, float16 and bfloat16 x."""
import ctypes

import numpy as np
import pytest
import torch

from gpu_util import check_matmul, quantized_layer, to_gpu
from oracle import rtn_oracle as orc

pytestmark = pytest.mark.gpu

FORMATS = [(4, 128), (4, 64), (4, 32), (8, 128), (8, 64), (8, 32), (2, 128), (2, 64), (2, 32)]


def _call(lib, x, d, n, bits, g, ldy, ws=True, bias=None):
    m, k = x.shape
    act = 0 if x.dtype is torch.float16 else 1
    y = torch.full((m, ldy), 7.0, dtype=torch.float16, device="cuda")
    need = lib.bw_qlinear_workspace_bytes(m, n, k, bits, g, act) if ws else 0
    w = torch.full((max(need, 16) // 4,), float("nan"), dtype=torch.float32, device="cuda")
    st = lib.bw_qlinear_ws(x.data_ptr(), act, m, k, x.stride(0), d[0].data_ptr(), d[1].data_ptr(), d[2].data_ptr(),
                           None if bias is None else bias.data_ptr(), n, bits, g, y.data_ptr(), ldy, w.data_ptr() if need else None, need,
                           ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    return st, y, need


@pytest.mark.parametrize("bits,g", FORMATS)
@pytest.mark.parametrize("k,n", [(128, 33), (23 * 128, 97), (9 * 64 * 2 + 64, 1003), (4096, 130)])
def test_rows_and_ragged_shapes_vs_oracle(bits, g, k, n):
    """K of one chunk, of an odd number of groups, not a multiple of 128 (or of 256), of several rounds; x rows padded and y rows of an
    odd pitch; with and without bias; with the workspace (K cut across workgroups on the narrow shapes) and without."""
    from bitween_amd.kernels import hip_loader
    lib = hip_loader.load()
    if k % g:
        k = k // g * g
    _, qw, s16, z16, b16 = quantized_layer(n, k, bits, g, seed=n + k + bits + g, outliers=True)
    w16 = orc.dequantize_f16(qw, s16, z16, g, bits)
    d = [to_gpu(a) for a in (qw, s16, z16, b16)]
    split = False
    for m in (17, 32, 33, 48, 64, 65, 96, 97, 128):
        gen = torch.Generator(device="cuda").manual_seed(m)
        xbuf = torch.full((m, k + 8), float("nan"), dtype=torch.float16, device="cuda")
        xbuf[:, :k] = torch.randn(m, k, device="cuda", generator=gen).half()
        hot = {0: k - 1, m - 1: k // 2}
        for r, c in hot.items():
            xbuf[r, :k] = 0
            xbuf[r, c] = 1.0
        x = xbuf[:, :k]
        st, y, need = _call(lib, x, d, n, bits, g, n + 1, bias=d[3])
        split = split or need > 0
        assert st == 0 and (y[:, n:] == 7.0).all()
        check_matmul(y[:, :n].contiguous(), x.cpu().numpy(), qw, s16, z16, b16, bits, g)
        st, y, _ = _call(lib, x, d, n, bits, g, n, ws=False)
        assert st == 0
        check_matmul(y, x.cpu().numpy(), qw, s16, z16, None, bits, g)
        for r, c in hot.items():
            assert np.array_equal(y[r].cpu().numpy().view(np.uint16), w16[:, c].view(np.uint16))
    assert split or k < 2048


@pytest.mark.parametrize("bits,g", FORMATS)
def test_bfloat16_rows_equal_the_cast(bits, g):
    """bfloat16 x is rounded to float16 as it is staged: the bits of a call on x.to(float16)."""
    from bitween_amd.kernels import hip_loader
    lib = hip_loader.load()
    n, k = 500, 1536
    _, qw, s16, z16, _ = quantized_layer(n, k, bits, g, seed=bits + g)
    d = [to_gpu(a) for a in (qw, s16, z16)]
    for m in (18, 40, 64, 80, 128):
        x = (torch.randn(m, k, device="cuda") * 30).to(torch.bfloat16)
        st, y, _ = _call(lib, x, d, n, bits, g, n)
        st2, y2, _ = _call(lib, x.to(torch.float16), d, n, bits, g, n)
        assert st == 0 and st2 == 0 and torch.equal(y, y2)


@pytest.mark.parametrize("bits,g,k,n", [(4, 64, 3072, 16400), (8, 32, 256, 12300), (2, 32, 4352, 4100), (4, 32, 8192, 200), (4, 128, 4224, 4100)])
@pytest.mark.parametrize("m", [5, 8, 9, 16])
def test_decode_rows_on_large_layers(bits, g, k, n, m):
    """Up to 16 rows the batch kernel takes layers with more column tiles, or longer rows, than the decode kernels stage once
    (and hands the others to them): through the module, and without a workspace."""
    from bitween_amd.kernels import hip_loader as hip
    rows = np.unique(np.concatenate([np.arange(0, n, n // 25), [n - 1]]))
    torch.manual_seed(m + k)
    lin = torch.nn.Linear(k, n, bias=True, device="cuda", dtype=torch.float16)
    import bitween_amd
    q = bitween_amd.QuantizedLinear.from_float(lin, bits, g)
    x = torch.randn(m, k, device="cuda", dtype=torch.float16)
    part = [a[torch.from_numpy(rows).cuda()].cpu().numpy() for a in (q.qweight, q.scale, q.zero_point, q.bias)]
    y = q(x)
    check_matmul(y[:, rows], x.cpu().numpy(), *part, bits, g)
    st, y2, _ = _call(hip.load(), x, (q.qweight, q.scale, q.zero_point), n, bits, g, n, ws=False, bias=q.bias)
    assert st == 0
    check_matmul(y2[:, rows], x.cpu().numpy(), *part, bits, g)
    xb = x.to(torch.bfloat16)
    assert torch.equal(q(xb), q(xb.to(torch.float16)))


@pytest.mark.parametrize("m", [7, 17, 70])
def test_layouts_the_batch_kernel_does_not_take(m):
    """Rows of x off a 16-byte boundary go to the generic kernel; scales off a 4-byte boundary do not, with bfloat16 x too; no x and an
    unknown type of x are refused."""
    from bitween_amd.kernels import hip_loader
    lib = hip_loader.load()
    bits, g, k, n = 4, 128, 1280, 260
    _, qw, s16, z16, b16 = quantized_layer(n, k, bits, g, seed=m)
    sbuf = torch.zeros(s16.size + 1, dtype=torch.float16, device="cuda")
    sbuf[1:] = to_gpu(s16).reshape(-1)
    s_odd = sbuf[1:].view(n, k // g)
    x = torch.randn(m, k, device="cuda", dtype=torch.float16)
    d = [to_gpu(qw), s_odd, to_gpu(z16)]
    st, y, _ = _call(lib, x, d, n, bits, g, n)
    assert st == 0
    check_matmul(y, x.cpu().numpy(), qw, s16, z16, None, bits, g)
    from bitween_amd.kernels import hip_loader as hip
    shifted = torch.empty(m, k + 8, device="cuda", dtype=torch.float16)[:, 1:k + 1]
    shifted.copy_(x)
    st, y, _ = _call(lib, shifted, d, n, bits, g, n)
    assert st == 0 and hip.last_decode_kernel() == ""
    check_matmul(y, x.cpu().numpy(), qw, s16, z16, None, bits, g)
    xb = x.to(torch.bfloat16)
    yb = hip.quantized_matmul_hip(xb, d[0], s_odd, d[2], to_gpu(b16), bits, g)
    check_matmul(yb, xb.to(torch.float16).cpu().numpy(), qw, s16, z16, b16, bits, g)
    assert lib.bw_qlinear_ws(None, 0, m, k, k, d[0].data_ptr(), d[1].data_ptr(), d[2].data_ptr(), None, n, bits, g, y.data_ptr(), n, None, 0, None) == -1
    assert lib.bw_qlinear_ws(x.data_ptr(), 2, m, k, k, d[0].data_ptr(), d[1].data_ptr(), d[2].data_ptr(), None, n, bits, g, y.data_ptr(), n, None, 0, None) == -2


@pytest.mark.parametrize("bits,g", FORMATS)
@pytest.mark.parametrize("m,k,n", [(129, 640, 1003), (333, 1152, 97), (500, 256, 515), (1025, 384, 130), (50, 512, 2050), (200, 4096, 66)])
def test_several_tiles_of_rows(bits, g, m, k, n):
    """More rows than a tile (or lower tiles than the call has rows): a last tile of one row, odd row counts, K cut across workgroups or
    not; rows of x and y padded, one-hot rows at the tiles' edges, every row against the oracle."""
    from bitween_amd.kernels import hip_loader
    lib = hip_loader.load()
    _, qw, s16, z16, b16 = quantized_layer(n, k, bits, g, seed=m + n + bits + g, outliers=True)
    w16 = orc.dequantize_f16(qw, s16, z16, g, bits)
    d = [to_gpu(a) for a in (qw, s16, z16, b16)]
    for dtype in (torch.float16, torch.bfloat16):
        xbuf = torch.full((m, k + 8), float("nan"), dtype=dtype, device="cuda")
        xbuf[:, :k] = torch.randn(m, k, device="cuda", generator=torch.Generator(device="cuda").manual_seed(m)).to(dtype)
        hot = {r: (37 * r) % k for r in (0, 15, 16, 31, 32, 47, 48, 63, 64, 95, 96, 127, 128, m - 1) if r < m}
        for r, c in hot.items():
            xbuf[r, :k] = 0
            xbuf[r, c] = 1.0
        x = xbuf[:, :k]
        for ws in (True, False):
            st, y, _ = _call(lib, x, d, n, bits, g, n + 1, ws=ws)
            if not ws and st == -5 and dtype is torch.bfloat16:      # the prefill kernel wants room for its cast
                continue
            assert st == 0 and (y[:, n:] == 7.0).all()
            check_matmul(y[:, :n].contiguous(), x.to(torch.float16).cpu().numpy(), qw, s16, z16, None, bits, g)
            for r, c in hot.items():
                assert np.array_equal(y[r, :n].cpu().numpy().view(np.uint16), w16[:, c].view(np.uint16))


@pytest.mark.parametrize("bits,g", FORMATS)
@pytest.mark.parametrize("m", [17, 40, 130])
def test_scales_off_a_four_byte_boundary(bits, g, m):
    """Row slices of scales and zero points with an odd number of groups may start inside a 4-byte word: the same kernel, so the same bits,
    as with arrays of their own (either array off the boundary, or both), for the first and the last group of every column."""
    from bitween_amd.kernels import hip_loader
    lib = hip_loader.load()
    n, k = 205, 9 * 128 + (g if g < 128 else 0)
    _, qw, s16, z16, b16 = quantized_layer(n, k, bits, g, seed=m + bits + g, outliers=True)
    qw, s, z, b = [to_gpu(a) for a in (qw, s16, z16, b16)]
    x = torch.randn(m, k, device="cuda", dtype=torch.float16)
    x[0], x[1] = 0, 0
    x[0, 0], x[1, k - 1] = 1, 1

    def shifted(t):
        buf = torch.full((t.numel() + 2,), float("nan"), dtype=t.dtype, device="cuda")
        buf[1:-1] = t.reshape(-1)
        return buf[1:-1].view(t.shape)

    st, want, _ = _call(lib, x, (qw, s, z), n, bits, g, n, bias=b)
    assert st == 0
    check_matmul(want, x.cpu().numpy(), qw.cpu().numpy(), s16, z16, b16, bits, g)
    for sv, zv in ((shifted(s), z), (s, shifted(z)), (shifted(s), shifted(z))):
        st, y, _ = _call(lib, x, (qw, sv, zv), n, bits, g, n, bias=b)
        assert st == 0 and torch.equal(y, want)


def test_last_kernel_names_the_batch_kernel_and_nothing_else():
    """bw_qgemv_last_kernel after each call of bw_qlinear_ws (with and without a workspace) and bw_qlinear: the decode or batch kernel of this
    very call, "" after the prefill and the generic kernel."""
    from bitween_amd.kernels import hip_loader as hip
    lib = hip.load()
    _, qw, s16, z16, _ = quantized_layer(272, 1024, 4, 128, seed=1)
    d = [to_gpu(a) for a in (qw, s16, z16)]

    def name(m, ws=True, dtype=torch.float16):
        st, _, _ = _call(lib, torch.randn(m, 1024, device="cuda").to(dtype), d, 272, 4, 128, 272, ws=ws)
        assert st == 0
        return hip.last_decode_kernel()

    decode = name(1)
    assert decode.startswith("qgemv_") and name(40).startswith("qbatch_kernel<4, 128, ") and name(1) == decode
    assert name(40, ws=False).startswith("qbatch_kernel<4, 128, ") and name(2100) == "" and name(1) == decode
    x = torch.randn(40, 1024, device="cuda", dtype=torch.float16)
    y = torch.empty(40, 272, device="cuda", dtype=torch.float16)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def qlinear(m, bits=4, g=128, k=1024, q=d):
        assert lib.bw_qlinear(x.data_ptr(), 0, m, k, 1024, q[0].data_ptr(), q[1].data_ptr(), q[2].data_ptr(), None, 272, bits, g, y.data_ptr(), 272, stream) == 0
        return hip.last_decode_kernel()

    assert qlinear(1) == decode and qlinear(40).startswith("q")
    _, qw, s16, z16, _ = quantized_layer(272, 960, 4, 48, seed=2)      # groups of 48: the generic kernel
    assert qlinear(3, g=48, k=960, q=[to_gpu(a) for a in (qw, s16, z16)]) == ""
    torch.cuda.synchronize()
