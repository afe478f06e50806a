"""The batch kernel's widest tiles, the order of its tiles on calls with many rows, and the lines between it and the decode kernels
up to 16 rows, against the oracle."""
import ctypes

import numpy as np
import pytest
import torch

from gpu_util import check_matmul
from test_gpu_batch import _call

pytestmark = pytest.mark.gpu


def _layer(n, k, bits, g):
    import bitween_amd
    torch.manual_seed(n + k)
    lin = torch.nn.Linear(k, n, bias=True, device="cuda", dtype=torch.float16)
    q = bitween_amd.QuantizedLinear.from_float(lin, bits, g)
    return (q.qweight, q.scale, q.zero_point), q.bias


def _check(x, d, bias, bits, g, columns, y):
    part = [a[torch.from_numpy(columns).cuda()].cpu().numpy() for a in (*d, bias)]
    check_matmul(y[:, torch.from_numpy(columns).cuda()], x.to(torch.float16).cpu().numpy(), *part, bits, g)


def _names_hold():
    """Plans and lines are counted in compute units; the kernel names of the cases below are those of 256."""
    return torch.cuda.get_device_properties(0).multi_processor_count == 256


def _tile(name):
    """(rows of 16, column tiles a wave) of a kernel name, qbatch_kernel<bits, group, rows, columns, ...>."""
    return tuple(int(p.rstrip(">")) for p in name.split(", ")[2:4])


def _columns(n, step=97):
    """A sample, with both ends and the edges of the 32-column tiles around them."""
    return np.unique(np.clip(np.concatenate([np.arange(0, n, step), [1, 15, 16, 31, 32, 63, 64, 127, 128], n - np.array([1, 2, 16, 17, 33])]), 0, n - 1))


@pytest.mark.parametrize("bits,g", [(4, 128), (4, 64), (4, 32), (2, 128), (2, 32)])
@pytest.mark.parametrize("m,n,k,tile", [(33, 8501, 256, (1, 4)), (17, 24751, 3200, (2, 4)), (45, 24751, 1152, (3, 4)), (260, 5501, 1024, (4, 4)),
                                        (128, 14336, 640, (8, 2))])
def test_four_column_tiles(bits, g, m, n, k, tile):
    """Layers wide enough for four column tiles a wave (the last: the widest plan of three rounds at 128 rows, eight row tiles and two): rows and
    columns that end inside a tile, one to three rounds of K, seven at 17 rows; bfloat16 x has the bits of its float16 cast."""
    from bitween_amd.kernels import hip_loader as hip
    d, bias = _layer(n, k, bits, g)
    gen = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn(m, k, device="cuda", generator=gen).to(torch.bfloat16)
    st, y, _ = _call(hip.load(), x.to(torch.float16), d, n, bits, g, n + 1, bias=bias)
    name = hip.last_decode_kernel()
    assert st == 0 and (y[:, n:] == 7.0).all() and name.startswith("qbatch_kernel<%d, %d, " % (bits, g))
    _check(x, d, bias, bits, g, _columns(n), y)
    st, yb, _ = _call(hip.load(), x, d, n, bits, g, n + 1, bias=bias)
    assert st == 0 and torch.equal(y, yb)
    if _names_hold():                                         # (W4 g128 scales sums of a group at 17 rows: at most 2 x 3 tiles do)
        assert _tile(name) == ((2, 2) if (bits, g, m) == (4, 128, 17) else tile), name


@pytest.mark.parametrize("bits,g", [(4, 128), (4, 64), (4, 32), (2, 128), (2, 64), (2, 32)])
@pytest.mark.parametrize("m,n,k,slices", [(128, 14336, 4096, 1), (113, 14325, 2560, 1), (122, 14325, 2048, 1), (97, 3967, 14336, 4), (64, 14325, 14336, 2)])
def test_four_by_four_tiles_in_their_loop(bits, g, m, n, k, slices):
    """64-row tiles of four column tiles a wave over many rounds of K: eight, five and four whole ones, seven of each of four slices, fourteen of
    each of two; bfloat16 x has the bits of its float16 cast."""
    from bitween_amd.kernels import hip_loader as hip
    d, bias = _layer(n, k, bits, g)
    x = torch.randn(m, k, device="cuda", generator=torch.Generator(device="cuda").manual_seed(m)).to(torch.bfloat16)
    st, y, need = _call(hip.load(), x.to(torch.float16), d, n, bits, g, n + 1, bias=bias)
    name = hip.last_decode_kernel()
    assert st == 0 and (y[:, n:] == 7.0).all()
    _check(x, d, bias, bits, g, _columns(n), y)
    st, yb, _ = _call(hip.load(), x, d, n, bits, g, n + 1, bias=bias)
    assert st == 0 and torch.equal(y, yb)
    if _names_hold():
        eight = (bits, g, m) == (4, 32, 97)                   # (there the spilled registers of W4 g32 cost the wide tile its place)
        assert _tile(name) == ((8, 2) if eight else (4, 4)) and need == (slices * m * -(-n // 4) * 4 * 4 if slices > 1 else 0), (name, need)


@pytest.mark.parametrize("bits,g,m,n,k", [(4, 128, 1100, 130, 1024), (4, 128, 700, 2050, 1664), (2, 64, 1030, 70, 4096), (8, 32, 620, 66, 2304),
                                          (4, 64, 530, 515, 2176), (4, 32, 257, 1030, 4192)])
def test_many_rows_every_tile_once(bits, g, m, n, k):
    """x beyond 2 MB in four and more tiles of rows, whose workgroups are numbered by XCD: panels of four and a shorter last one, grids that
    are no multiple of eight, K cut or not; nothing is left out and nothing beyond y is written."""
    from bitween_amd.kernels import hip_loader as hip
    d, bias = _layer(n, k, bits, g)
    x = torch.randn(m, k, device="cuda", generator=torch.Generator(device="cuda").manual_seed(m)).to(torch.float16)
    assert m * k * 2 > 2 << 20
    st, y, _ = _call(hip.load(), x, d, n, bits, g, n + 3, bias=bias)
    assert st == 0 and (y[:, n:] == 7.0).all() and hip.last_decode_kernel().startswith("qbatch_kernel<")
    _check(x, d, bias, bits, g, np.arange(n) if n < 200 else _columns(n, 23), y)


@pytest.mark.parametrize("bits,g,m,n,k,ldx", [(4, 64, 300, 530, 1024, 4096), (4, 128, 260, 1030, 1024, 5120), (2, 64, 300, 530, 2048, 4104)])
def test_padded_rows_in_the_order_by_xcd(bits, g, m, n, k, ldx):
    """The order of the workgroups hangs on the extent of x, its pitch included: rows of a wider buffer go past 2 MB where their values would not,
    and give the bits of the same rows side by side."""
    from bitween_amd.kernels import hip_loader as hip
    d, bias = _layer(n, k, bits, g)
    assert m * k * 2 <= 2 << 20 < ((m - 1) * ldx + k) * 2
    for dtype in (torch.float16, torch.bfloat16):
        wide = torch.full((m, ldx), float("nan"), device="cuda", dtype=dtype)
        wide[:, :k] = torch.randn(m, k, device="cuda", generator=torch.Generator(device="cuda").manual_seed(m))
        st, y, _ = _call(hip.load(), wide[:, :k], d, n, bits, g, n + 3, bias=bias)
        assert st == 0 and (y[:, n:] == 7.0).all() and hip.last_decode_kernel().startswith("qbatch_kernel<")
        _check(wide[:, :k], d, bias, bits, g, _columns(n, 23), y)
        st, dense, _ = _call(hip.load(), wide[:, :k].contiguous(), d, n, bits, g, n + 3, bias=bias)
        assert st == 0 and torch.equal(y, dense)


@pytest.mark.parametrize("bits,g,k,n,m,kernel", [
    (4, 128, 10368, 2048, 9, "qbatch"), (4, 128, 10240, 2048, 16, "qgemv"), (4, 128, 10368, 2048, 8, "qgemv"), (4, 128, 10368, 2064, 16, "qgemv"),
    (4, 128, 4224, 4112, 5, "qbatch"), (4, 128, 4096, 4112, 16, "qgemv"), (4, 64, 11072, 2064, 9, "qbatch"), (4, 64, 11008, 2064, 9, "qgemv"),
    (4, 32, 544, 4112, 9, "qbatch"), (4, 32, 544, 4096, 9, "qgemv"), (4, 32, 9248, 640, 5, "qbatch"), (4, 32, 9216, 640, 5, "qgemv"), (4, 64, 11328, 512, 5, "qbatch"), (4, 64, 11264, 512, 8, "qgemv"),
    (2, 64, 12352, 512, 5, "qbatch"), (2, 64, 12288, 512, 8, "qgemv"), (2, 64, 8256, 1024, 9, "qbatch"), (2, 128, 8192, 1024, 16, "qgemv"),
    (8, 32, 6432, 1024, 9, "qbatch"), (8, 32, 6400, 1024, 9, "qgemv"), (2, 128, 8320, 2064, 12, "qbatch"),
    (4, 128, 1024, 12304, 9, "qbatch"), (4, 128, 4096, 12304, 9, "qgemv"), (4, 128, 3968, 12304, 9, "qbatch"),
    (2, 128, 8448, 4096, 9, "qgemv"), (2, 128, 8320, 4096, 9, "qbatch"),
    (2, 64, 12288, 4096, 9, "qgemv"), (2, 64, 12416, 4096, 9, "qbatch"), (4, 64, 13312, 4096, 9, "qgemv"), (4, 64, 13440, 4096, 9, "qbatch"),
    (2, 64, 3072, 12304, 16, "qbatch"), (2, 64, 3200, 12304, 16, "qgemv"), (8, 128, 3200, 4112, 16, "qbatch"), (8, 128, 3072, 4112, 16, "qgemv"), (8, 128, 3200, 4112, 8, "qgemv"),
    (8, 128, 8192, 2048, 9, "qbatch"), (8, 32, 8224, 640, 5, "qbatch"), (8, 64, 8192, 2064, 9, "qbatch"), (8, 64, 8128, 2064, 9, "qgemv"),
    (8, 64, 1088, 12304, 9, "qbatch"), (8, 64, 1024, 12304, 9, "qgemv"), (8, 64, 3136, 16384, 6, "qbatch"), (8, 64, 3072, 16384, 6, "qgemv"),
    (8, 64, 3136, 16400, 6, "qgemv")])
def test_lines_between_decode_and_batch_rows(bits, g, k, n, m, kernel):
    """5 ... 16 rows on both sides of each line (256 compute units), K cut across workgroups where the layer is narrow; a narrow layer's
    call without a workspace for that cut stays with the decode kernels."""
    from bitween_amd.kernels import hip_loader as hip
    d, bias = _layer(n, k, bits, g)
    x = torch.randn(m, k, device="cuda", generator=torch.Generator(device="cuda").manual_seed(m)).to(torch.float16)
    st, y, need = _call(hip.load(), x, d, n, bits, g, n, bias=bias)
    name = hip.last_decode_kernel()
    assert st == 0
    _check(x, d, bias, bits, g, _columns(n), y)
    st, y, _ = _call(hip.load(), x, d, n, bits, g, n, ws=False, bias=bias)
    uncut = hip.last_decode_kernel()
    assert st == 0
    _check(x, d, bias, bits, g, _columns(n), y)
    if _names_hold():
        assert name.startswith(kernel) and uncut.startswith("qgemv" if need and n <= 4096 else kernel)


@pytest.mark.parametrize("bits,g,m,n,k", [(4, 128, 813, 4432, 2304), (4, 64, 200, 9000, 6912), (2, 64, 1167, 3340, 1024), (8, 32, 1171, 3842, 1024)])
def test_bfloat16_without_room_for_its_cast(bits, g, m, n, k):
    """Calls that the prefill kernel is expected to finish first, with bfloat16 x: with no workspace, and with 16 bytes less than the cast takes,
    the batch kernel runs them (and writes nothing beyond the workspace); beyond 2048 rows there is none that could."""
    from bitween_amd.kernels import hip_loader as hip
    lib = hip.load()
    d, bias = _layer(n, k, bits, g)
    x = torch.randn(m, k, device="cuda", generator=torch.Generator(device="cuda").manual_seed(m)).to(torch.bfloat16)
    st, y, need = _call(lib, x, d, n, bits, g, n, bias=bias)
    if _names_hold():
        assert hip.last_decode_kernel() == "" and need >= 2 * m * k
    _check(x, d, bias, bits, g, _columns(n), y)
    short = 2 * m * k - 16
    ws = torch.full((short + 64,), 85, dtype=torch.uint8, device="cuda")
    y = torch.full((m, n), 7.0, dtype=torch.float16, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for buffer, size in ((None, 0), (ws.data_ptr(), short)):
        y.fill_(7.0)
        st = lib.bw_qlinear_ws(x.data_ptr(), 1, m, k, k, d[0].data_ptr(), d[1].data_ptr(), d[2].data_ptr(), bias.data_ptr(), n, bits, g, y.data_ptr(), n,
                               buffer, size, stream)
        torch.cuda.synchronize()
        assert st == 0 and hip.last_decode_kernel().startswith("qbatch_kernel<%d, %d, " % (bits, g)) and (ws[short:] == 85).all()
        _check(x, d, bias, bits, g, _columns(n), y)
    x = torch.zeros(2050, k, dtype=torch.bfloat16, device="cuda")
    y = torch.zeros(2050, n, dtype=torch.float16, device="cuda")
    assert lib.bw_qlinear_ws(x.data_ptr(), 1, 2050, k, k, d[0].data_ptr(), d[1].data_ptr(), d[2].data_ptr(), None, n, bits, g, y.data_ptr(), n, None, 0, stream) == -5
