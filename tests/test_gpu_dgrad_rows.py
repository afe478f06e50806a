"""The input gradient of a few rows (weights unpacked to operand layout without a way through LDS) against the oracle: every format, both
gradient types and each number of row tiles, rows and n that end inside a tile, a step or a wave's turn, strips of K that end inside 256 columns,
and the calls that keep the other kernels for their alignment."""
import ctypes

import numpy as np
import pytest
import torch

from gpu_util import quantized_layer, to_gpu
from oracle import rtn_oracle as orc
from test_gpu_dgrad import COMBOS, _check

pytestmark = pytest.mark.gpu


def _call(go, d, n, k, bits, g, ldg, scale_off=0):
    from bitween_amd.kernels import hip_loader
    lib = hip_loader.load()
    m = go.shape[0]
    buf = torch.full((m, ldg), float("nan"), dtype=go.dtype, device="cuda")     # the padding must never be read
    buf[:, :n] = go
    need = lib.bw_qdgrad_workspace_bytes(m, n, k, bits, g)
    ws = torch.full((need + 4096,), 85, dtype=torch.uint8, device="cuda")
    gx = torch.full((m, k + 4), 7.0, dtype=go.dtype, device="cuda")
    scale = torch.zeros(d[1].numel() + scale_off, dtype=torch.float16, device="cuda")
    scale[scale_off:] = d[1].reshape(-1)
    st = lib.bw_qdgrad(buf.data_ptr(), int(go.dtype == torch.bfloat16), m, n, ldg, d[0].data_ptr(), scale.data_ptr() + 2 * scale_off, d[2].data_ptr(), k, bits, g,
                       gx.data_ptr(), k + 4, ws.data_ptr(), need, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert st == 0 and (ws[need:] == 85).all() and (gx[:, k:] == 7.0).all()
    return gx[:, :k]


@pytest.mark.parametrize("bits,g", COMBOS)
@pytest.mark.parametrize("n,k", [(6248, 1024), (2824, 2304 + 256)])
def test_rows_vs_oracle(bits, g, n, k):
    _, qw, s16, z16, _ = quantized_layer(n, k, bits, g, seed=n + k + bits + g, outliers=True, bias=False)
    d = [to_gpu(a) for a in (qw, s16, z16)]
    rng = np.random.default_rng(n + bits)
    wb = orc.dequantize_bf16(qw, s16, z16, g, bits)
    for m in (1, 7, 16, 17, 32):
        go16 = rng.standard_normal((m, n)).astype(np.float16)
        hot = {0: n - 1, m // 2: 0, m - 1: n // 2 + 1}
        for r, c in hot.items():
            go16[r] = 0
            go16[r, c] = 1
        gx = _call(to_gpu(go16), d, n, k, bits, g, n + 8)
        _check(gx, go16, qw, s16, z16, bits, g)
        w16 = orc.dequantize_f16(qw, s16, z16, g, bits)
        for r, c in hot.items():
            assert np.array_equal(gx[r].cpu().numpy(), w16[c])
        gob = to_gpu(go16).to(torch.bfloat16)
        gb = _call(gob, d, n, k, bits, g, n + 8)
        want = gob.double().cpu().numpy() @ np.asarray(wb, dtype=np.float64)
        # one rounding to bfloat16 and float32 sums
        bound = 2.0 ** -8 * np.abs(want) + 2e-6 * (np.abs(gob.double().cpu().numpy()) @ np.abs(np.asarray(wb, dtype=np.float64))) + 1e-7
        assert (np.abs(gb.double().cpu().numpy() - want) <= bound).all()
        for r, c in hot.items():
            assert np.array_equal(gb[r].float().cpu().numpy(), np.asarray(wb[c], dtype=np.float32))


@pytest.mark.parametrize("bits,g,n,k", [(4, 32, 4160, 1088), (8, 32, 2048, 2112), (2, 64, 3016, 1408)])
def test_strips_of_columns_that_end_early(bits, g, n, k):
    _, qw, s16, z16, _ = quantized_layer(n, k, bits, g, seed=n + k, outliers=True, bias=False)
    d = [to_gpu(a) for a in (qw, s16, z16)]
    go16 = np.random.default_rng(k).standard_normal((11, n)).astype(np.float16)
    _check(_call(to_gpu(go16), d, n, k, bits, g, n), go16, qw, s16, z16, bits, g)


@pytest.mark.parametrize("n,k,ldg,scale_off", [(6252, 1024, 6256, 0), (6248, 1024, 6250, 0), (6248, 1024, 6248, 1), (4096, 1152, 4096, 0)])
def test_calls_that_keep_the_other_kernels(n, k, ldg, scale_off):
    """n off eights, rows of the gradient off 16 bytes, scales off four bytes, an odd number of groups."""
    bits, g = 4, 128
    _, qw, s16, z16, _ = quantized_layer(n, k, bits, g, seed=n + k, outliers=True, bias=False)
    d = [to_gpu(a) for a in (qw, s16, z16)]
    go16 = np.random.default_rng(n).standard_normal((9, n)).astype(np.float16)
    _check(_call(to_gpu(go16), d, n, k, bits, g, ldg, scale_off), go16, qw, s16, z16, bits, g)


@pytest.mark.parametrize("bits,g", COMBOS)
def test_two_and_three_row_tiles_of_large_layers(bits, g):
    """bfloat16 gradients of 17 ... 32 rows and float16 gradients of 33 ... 48 come here from 30 (8 bits: 40) million weights on: every format, n that ends
    inside a step, and where groups allow it K inside a strip.  That this kernel ran shows in the workspace, of which it fills its own slices."""
    import bitween_amd
    from bitween_amd.kernels import hip_loader
    lib = hip_loader.load()
    n, k = 9784, 4096 + (2 * g if g < 128 else 0)
    torch.manual_seed(bits * g)
    q = bitween_amd.QuantizedLinear.from_float(torch.nn.Linear(k, n, bias=False, device="cuda", dtype=torch.float16), bits, g)
    arrays = [t.cpu().numpy() for t in (q.qweight, q.scale, q.zero_point)]
    w16, wb = (np.asarray(f(*arrays, g, bits), dtype=np.float64) for f in (orc.dequantize_f16, orc.dequantize_bf16))
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for dtype, code, m in ((torch.bfloat16, 1, 17), (torch.bfloat16, 1, 32), (torch.float16, 0, 33), (torch.float16, 0, 48)):
        w, ulp = (wb, 2.0 ** -8) if code else (w16, 2.0 ** -11)
        go = torch.randn(m, n, device="cuda").to(dtype)
        hot = {0: n - 1, m - 1: 31}
        for r, c in hot.items():
            go[r] = 0
            go[r, c] = 1
        slices, need = lib.bw_qdgrad_rows_slices(m, n, k, bits, g, code), lib.bw_qdgrad_workspace_bytes(m, n, k, bits, g)
        assert slices > 1
        ws = torch.full((need,), 85, dtype=torch.uint8, device="cuda")
        gx = torch.empty(m, k, dtype=dtype, device="cuda")
        assert lib.bw_qdgrad(go.data_ptr(), code, m, n, n, q.qweight.data_ptr(), q.scale.data_ptr(), q.zero_point.data_ptr(), k, bits, g, gx.data_ptr(), k,
                             ws.data_ptr(), need, stream) == 0
        torch.cuda.synchronize()
        words = ws[:need // 4 * 4].view(torch.int32) == 0x55555555
        own = slices * m * k
        assert not words[:own].any() and words[own:].all()
        g64 = go.double().cpu().numpy()
        want = g64 @ w
        bound = ulp * np.abs(want) + 2e-6 * (np.abs(g64) @ np.abs(w)) + 1e-7   # one rounding and float32 sums
        got = gx.double().cpu().numpy()
        assert (np.abs(got - want) <= bound).all()
        for r, c in hot.items():
            assert np.array_equal(got[r], w[c])


@pytest.mark.parametrize("bits,g,m,n,k", [(8, 32, 8, 8752, 4864), (4, 64, 17, 8752, 2176)])
def test_partial_tiles_of_the_stepping_kernel_on_large_layers(bits, g, m, n, k):
    """Rows of the gradient off 16 bytes keep the stepping kernel, also where the kernel of a few rows would take the layer: its partial tiles are the call's
    rows high and stay inside the workspace."""
    from bitween_amd.kernels import hip_loader
    assert hip_loader.load().bw_qdgrad_rows_slices(m, n, k, bits, g, 0) > 0       # (with rows on 16 bytes)
    _, qw, s16, z16, _ = quantized_layer(n, k, bits, g, seed=n + k, outliers=True, bias=False)
    d = [to_gpu(a) for a in (qw, s16, z16)]
    go16 = np.random.default_rng(m).standard_normal((m, n)).astype(np.float16)
    _check(_call(to_gpu(go16), d, n, k, bits, g, n + 2), go16, qw, s16, z16, bits, g)


def test_three_row_tiles_and_infinities():
    """33 ... 48 rows of a large layer; an infinity stays in its row."""
    bits, g, n, k, m = 4, 128, 7680, 4096, 41
    _, qw, s16, z16, _ = quantized_layer(n, k, bits, g, seed=5, outliers=True, bias=False)
    d = [to_gpu(a) for a in (qw, s16, z16)]
    go16 = np.random.default_rng(6).standard_normal((m, n)).astype(np.float16)
    _check(_call(to_gpu(go16), d, n, k, bits, g, n), go16, qw, s16, z16, bits, g)
    inf = go16.copy()
    inf[40, n - 1] = np.inf
    inf[3, 0] = -np.inf
    a, b = _call(to_gpu(go16), d, n, k, bits, g, n), _call(to_gpu(inf), d, n, k, bits, g, n)
    rest = [r for r in range(m) if r not in (3, 40)]
    assert torch.equal(a[rest], b[rest]) and not torch.isfinite(b[[3, 40]]).any()
