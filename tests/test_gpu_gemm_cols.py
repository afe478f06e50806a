"""The prefill kernel's tiles - 192 columns (three column tiles a wave) and 256 - against the oracle: forced through the measurement build, which takes
the tile from the environment, and, every format on every tile, as the library itself chooses them (the kernel's waits are counted by hand around
assembly: what has been compiled is what has to be run)."""
import ctypes

import numpy as np
import pytest
import torch

from gpu_util import check_matmul, quantized_layer, to_gpu
from oracle import rtn_oracle as orc

pytestmark = pytest.mark.gpu

FORMATS = [(4, 128), (4, 64), (4, 32), (8, 128), (8, 64), (8, 32), (2, 128), (2, 64), (2, 32)]


def _forced(monkeypatch, rows, cols):
    from bitween_amd.csrc import build
    from bitween_amd.kernels import hip_loader
    lib, ref = ctypes.CDLL(build.TUNE_LIB), hip_loader.load()
    for name in ("bw_qgemm_ws", "bw_qgemm_workspace_bytes"):
        fn = getattr(lib, name)
        fn.argtypes, fn.restype = getattr(ref, name).argtypes, getattr(ref, name).restype
    monkeypatch.setenv("BW_GEMM_BM", str(rows))
    monkeypatch.setenv("BW_GEMM_BN", str(cols))
    return lib


def _run(lib, x, d, bias, n, bits, g, ldy, with_workspace=False):
    m, k = x.shape
    y = torch.full((m, ldy), 7.0, dtype=torch.float16, device="cuda")
    need = lib.bw_qgemm_workspace_bytes(m, n, k, bits, g) if with_workspace else 0
    ws = torch.empty(max(need, 16), dtype=torch.uint8, device="cuda")
    st = lib.bw_qgemm_ws(x.data_ptr(), 0, m, k, k, *[t.data_ptr() for t in d], bias.data_ptr() if bias is not None else None, n, bits, g,
                         y.data_ptr(), ldy, ws.data_ptr() if need else None, need, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert st == 0
    torch.cuda.synchronize()
    assert (y[:, n:] == 7.0).all()
    return y[:, :n]


@pytest.mark.parametrize("rows", [128, 256])
@pytest.mark.parametrize("bits,g", FORMATS)
@pytest.mark.parametrize("k,n,m,pad", [(128, 191, 129, 1), (256, 193, 257, 7), (384, 48, 130, 0), (640, 400, 200, 0), (896, 239, 300, 1), (1024, 576, 513, 8)])
def test_192_column_tiles(monkeypatch, rows, bits, g, k, n, m, pad):
    """One to eight K steps (odd counts, runs of four and what is left of them), columns that end in every quarter of a tile and inside a
    wave's 48, rows past a tile, rows of y on and off 16 bytes; one-hot rows return columns of W16 bit for bit."""
    lib = _forced(monkeypatch, rows, 192)
    _, qw, s16, z16, b16 = quantized_layer(n, k, bits, g, seed=k + n + g + bits, outliers=True)
    x = np.random.default_rng(m).standard_normal((m, k)).astype(np.float16)
    d = [to_gpu(a) for a in (qw, s16, z16)]
    check_matmul(_run(lib, to_gpu(x), d, to_gpu(b16), n, bits, g, n + pad), x, qw, s16, z16, b16, bits, g)
    cols = np.linspace(0, k - 1, m).astype(int)
    hot = np.zeros((m, k), np.float16)
    hot[np.arange(m), cols] = 1
    y = _run(lib, to_gpu(hot), d, None, n, bits, g, n + pad)
    assert np.array_equal(y.cpu().numpy(), orc.dequantize_f16(qw, s16, z16, g, bits)[:, cols].T)


@pytest.mark.parametrize("rows", [128, 256])
@pytest.mark.parametrize("bits,g", [(4, 128), (8, 32), (2, 64)])
def test_192_column_tiles_cut_along_k(monkeypatch, rows, bits, g):
    """Partial tiles of 192 columns and their sum: slices of whole pairs of K steps and a shorter last one."""
    n, k, m = 401, 128 * 22, 300
    lib = _forced(monkeypatch, rows, 192)
    assert lib.bw_qgemm_workspace_bytes(m, n, k, bits, g) > 0
    _, qw, s16, z16, b16 = quantized_layer(n, k, bits, g, seed=rows + g, outliers=True)
    x = np.random.default_rng(rows).standard_normal((m, k)).astype(np.float16)
    d = [to_gpu(a) for a in (qw, s16, z16)]
    check_matmul(_run(lib, to_gpu(x), d, to_gpu(b16), n, bits, g, n + 3, with_workspace=True), x, qw, s16, z16, b16, bits, g)


@pytest.mark.parametrize("rows", [64, 128, 256])
@pytest.mark.parametrize("bits,g", FORMATS)
@pytest.mark.parametrize("k,n,m,pad", [(128, 255, 65, 1), (256, 257, 257, 7), (384, 64, 130, 0), (640, 400, 200, 0), (896, 301, 300, 1), (1024, 576, 513, 8)])
def test_256_column_tiles(monkeypatch, rows, bits, g, k, n, m, pad):
    """The same for 256 columns, which small calls have given up to the narrower tiles: 8 bits hands weights over between lanes here too (64 and
    128 rows; in groups of 32 the scales as well)."""
    lib = _forced(monkeypatch, rows, 256)
    _, qw, s16, z16, b16 = quantized_layer(n, k, bits, g, seed=k + n + g + bits, outliers=True)
    x = np.random.default_rng(m).standard_normal((m, k)).astype(np.float16)
    d = [to_gpu(a) for a in (qw, s16, z16)]
    check_matmul(_run(lib, to_gpu(x), d, to_gpu(b16), n, bits, g, n + pad), x, qw, s16, z16, b16, bits, g)
    cols = np.linspace(0, k - 1, m).astype(int)
    hot = np.zeros((m, k), np.float16)
    hot[np.arange(m), cols] = 1
    y = _run(lib, to_gpu(hot), d, None, n, bits, g, n + pad)
    assert np.array_equal(y.cpu().numpy(), orc.dequantize_f16(qw, s16, z16, g, bits)[:, cols].T)


@pytest.mark.parametrize("rows", [64, 128])
@pytest.mark.parametrize("g", [32, 64, 128])
def test_256_column_tiles_of_8_bits_cut_along_k(monkeypatch, rows, g):
    bits, n, k, m = 8, 401, 128 * 22, 300
    lib = _forced(monkeypatch, rows, 256)
    assert lib.bw_qgemm_workspace_bytes(m, n, k, bits, g) > 0
    _, qw, s16, z16, b16 = quantized_layer(n, k, bits, g, seed=rows + g, outliers=True)
    x = np.random.default_rng(rows).standard_normal((m, k)).astype(np.float16)
    d = [to_gpu(a) for a in (qw, s16, z16)]
    check_matmul(_run(lib, to_gpu(x), d, to_gpu(b16), n, bits, g, n + 3, with_workspace=True), x, qw, s16, z16, b16, bits, g)


# rows, columns of the tile: calls that get it for some K of the list below (256 compute units), and whether K is cut
TILES = [(64, 256, [(65, 301), (113, 517)]), (128, 192, [(139, 301), (80, 4505)]), (128, 256, [(1400, 197), (816, 194), (1200, 203), (69, 9721), (66, 5840)]),
         (256, 192, [(1900, 9601), (2213, 8223), (2743, 6607)]), (256, 256, [(1180, 9860), (1060, 11078), (2563, 4654), (2907, 4511), (1159, 9877)])]


@pytest.mark.parametrize("bits,g", FORMATS)
@pytest.mark.parametrize("rows,cols,calls", TILES, ids=["%dx%d" % t[:2] for t in TILES])
def test_every_tile_of_the_library_itself(rows, cols, calls, bits, g):
    """The first call of the list that gets the tile with more than two K steps, else with two: one-hot rows return columns of W16 bit for bit,
    random rows agree with the library product of W16 everywhere and with the oracle on samples."""
    from bitween_amd.kernels import hip_loader
    lib = hip_loader.load()
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("which tile a call gets depends on the number of compute units")
    picked = [(m, n, k) for k in (1152, 640, 384, 2560, 3072, 4096, 256) for m, n in calls
              if (lib.bw_qgemm_tile_rows(m, n, k, bits, g), lib.bw_qgemm_tile_cols(m, n, k, bits, g)) == (rows, cols)]
    assert picked, "no call of the list has this tile any more"
    m, n, k = picked[0]
    _, qw, s16, z16, b16 = quantized_layer(n, k, bits, g, seed=m + n + g, outliers=True)
    d = [to_gpu(a) for a in (qw, s16, z16)]
    w16 = to_gpu(orc.dequantize_f16(qw, s16, z16, g, bits))
    at = torch.linspace(0, k - 1, m).long().cuda()
    hot = torch.zeros(m, k, dtype=torch.float16, device="cuda")
    hot[torch.arange(m, device="cuda"), at] = 1
    assert torch.equal(_run(lib, hot, d, None, n, bits, g, n + 1, with_workspace=True), w16[:, at].T)
    x = torch.randn(m, k, device="cuda").half()
    y = _run(lib, x, d, to_gpu(b16), n, bits, g, n, with_workspace=True)
    ref = (x @ w16.T).float() + to_gpu(b16).float()
    assert ((y.float() - ref).abs().max() <= 2.0 ** -8 * ref.abs().max()).item()
    sample = torch.unique(torch.cat([torch.arange(0, m, max(1, m // 24)), torch.arange(m - 3, m)]))
    check_matmul(y[sample.cuda()], x[sample.cuda()].cpu().numpy(), qw, s16, z16, b16, bits, g)


@pytest.mark.parametrize("bits,g,m,n,k", [(8, 32, 509, 11008, 4096), (4, 128, 1000, 11008, 4096), (4, 64, 160, 6000, 2048)])
def test_tiles_the_library_chooses(bits, g, m, n, k):
    """Columns at the edges of the 192- and 256-column tiles."""
    import bitween_amd
    from bitween_amd.kernels import hip_loader
    lib = hip_loader.load()
    torch.manual_seed(n)
    q = bitween_amd.QuantizedLinear.from_float(torch.nn.Linear(k, n, bias=True, device="cuda", dtype=torch.float16), bits, g)
    x = torch.randn(m, k, device="cuda", dtype=torch.float16)
    y = _run(lib, x, (q.qweight, q.scale, q.zero_point), q.bias, n, bits, g, n, with_workspace=True)
    cols = np.unique(np.clip(np.concatenate([np.arange(0, n, 331)] + [e + np.arange(-1, 2) for e in (48, 64, 192, 256, n - n % 192, n)]), 0, n - 1))
    part = [t[torch.from_numpy(cols).cuda()].cpu().numpy() for t in (q.qweight, q.scale, q.zero_point, q.bias)]
    check_matmul(y[:, torch.from_numpy(cols).cuda()], x.cpu().numpy(), *part, bits, g)


@pytest.mark.parametrize("m,n,k", [(1255, 4656, 12160), (467, 12000, 11904), (300, 4096, 4096)])
def test_the_librarys_own_array_runs_the_same_plan(m, n, k):
    """bw_qgemm_static gives the bits of bw_qgemm_ws with all the workspace it asks for: no plan of 192-column tiles needs more than the 32 MiB array
    (the first two would, with 256 rows, and were accepted before)."""
    import bitween_amd
    from bitween_amd.kernels import hip_loader
    lib = hip_loader.load()
    q = bitween_amd.QuantizedLinear.from_float(torch.nn.Linear(k, n, bias=True, device="cuda", dtype=torch.float16), 4, 128)
    x = torch.randn(m, k, device="cuda", dtype=torch.float16)
    y = _run(lib, x, (q.qweight, q.scale, q.zero_point), q.bias, n, 4, 128, n, with_workspace=True)
    z = torch.empty_like(y)
    st = lib.bw_qgemm_static(x.data_ptr(), 0, m, k, k, q.qweight.data_ptr(), q.scale.data_ptr(), q.zero_point.data_ptr(), q.bias.data_ptr(), n, 4, 128,
                             z.data_ptr(), n, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert st == 0 and torch.equal(y, z)


@pytest.mark.parametrize("m,n,k,bits,g,cuts", [(1287, 2000, 6016, 4, 128, True), (98, 9472, 6272, 8, 32, True), (339, 7376, 2688, 4, 64, False),
                                                  (227, 11728, 2688, 4, 64, False)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_a_workspace_smaller_than_asked_for(m, n, k, bits, g, cuts, dtype):
    """bw_qlinear_ws with 16 bytes less than the chosen plan of 192-column tiles asks for: the cut plan of the 256-column tiles runs where it is expected to
    be done before the uncut ones (then bit for bit bw_qgemm_ws's), else the uncut one, which leaves the workspace alone."""
    import bitween_amd
    from bitween_amd.kernels import hip_loader
    lib = hip_loader.load()
    if torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the plans depend on the number of compute units")
    torch.manual_seed(k)
    q = bitween_amd.QuantizedLinear.from_float(torch.nn.Linear(k, n, bias=True, device="cuda", dtype=torch.float16), bits, g)
    x = torch.randn(m, k, device="cuda").to(dtype)
    bf16 = int(dtype == torch.bfloat16)
    full = lib.bw_qlinear_workspace_bytes(m, n, k, bits, g, bf16)
    cast = full - lib.bw_qgemm_workspace_bytes(m, n, k, bits, g)
    assert cast == (-(-m * k * 2 // 256) * 256 if bf16 else 0), "case is meant to run on the prefill kernel"
    args = [t.data_ptr() for t in (q.qweight, q.scale, q.zero_point, q.bias)]
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    y, z = (torch.empty(m, n, dtype=torch.float16, device="cuda") for _ in range(2))
    ws, other = (torch.full((full,), 85, dtype=torch.uint8, device="cuda") for _ in range(2))
    assert lib.bw_qlinear_ws(x.data_ptr(), bf16, m, k, k, *args, n, bits, g, y.data_ptr(), n, ws.data_ptr(), full - 16, st) == 0
    x16 = x.half()
    assert lib.bw_qgemm_ws(x16.data_ptr(), 0, m, k, k, *args, n, bits, g, z.data_ptr(), n, other.data_ptr() if cuts else None, full - cast - 16 if cuts else 0, st) == 0
    torch.cuda.synchronize()
    assert torch.equal(y, z) and (ws[full - 16:] == 85).all()
    assert (ws[cast:] == 85).all().item() != cuts
    cols = np.unique(np.linspace(0, n - 1, 60).astype(int))
    part = [t[torch.from_numpy(cols).cuda()].cpu().numpy() for t in (q.qweight, q.scale, q.zero_point, q.bias)]
    check_matmul(y[:, torch.from_numpy(cols).cuda()], x16.cpu().numpy(), *part, bits, g)
