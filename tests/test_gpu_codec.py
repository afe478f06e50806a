"""Quantise and dequantise where their launches change shape: the loads that a wave shares through LDS (from 4 M weights on),
whose last wave of a row may be partly past the row's end, and the 16-byte pieces of the output, flat or with padded rows."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

CODE = {torch.float16: 0, torch.bfloat16: 1, torch.float32: 2}


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


@pytest.mark.parametrize("with_delta", [False, True])
@pytest.mark.parametrize("dtype,bits,g,k", [(torch.float32, 4, 128, 4096), (torch.float32, 2, 32, 4192), (torch.float32, 8, 16, 1040),
                                            (torch.float16, 8, 32, 2080), (torch.bfloat16, 8, 64, 4160)])
def test_shared_loads_give_the_same_words(dtype, bits, g, k, with_delta):
    """Rows quantised together (4 M weights and more) and in parts too small for the shared loads: the same words, scales and zero
    points, bit for bit (a row's result depends on nothing but the row).  The small parts are what the oracle tests cover."""
    from bitween_amd.kernels import hip_loader as hip
    n = (4 << 20) // k + 3
    torch.manual_seed(k)
    w = torch.randn(n, k, device="cuda").to(dtype)
    delta = (0.01 * torch.randn(n, k, device="cuda")).to(dtype) if with_delta else None
    whole = hip.quantize_pack(w, bits, g, torch.float32, torch.float32, torch.int32, delta=delta)
    for r in range(0, n, n // 3):
        part = hip.quantize_pack(w[r:r + n // 3], bits, g, torch.float32, torch.float32, torch.int32,
                                 delta=None if delta is None else delta[r:r + n // 3])
        for a, b in zip(whole, part):
            assert torch.equal(a[r:r + n // 3], b)


@pytest.mark.parametrize("pad", [0, 8])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("bits,g,n,k", [(2, 32, 5, 96), (4, 16, 3, 80), (8, 8, 7, 72), (4, 128, 33, 1152), (8, 256, 2, 256),
                                        (2, 64, 2200, 16384)])            # the last: 134 MiB of float32 leave with the non-temporal hint
def test_dequantize_pieces(bits, g, n, k, dtype, pad):
    """scale * (q - zero_point), one rounding each and one to the output's type; padding between rows stays as it was."""
    from bitween_amd.kernels import hip_loader as hip
    lib = hip.load()
    torch.manual_seed(n)
    words = torch.randint(-2 ** 31, 2 ** 31, (n, k * bits // 32), dtype=torch.int64, device="cuda").to(torch.int32)
    scale = 0.01 + torch.rand(n, k // g, device="cuda")
    zero = torch.randint(0, 2 ** bits, (n, k // g), dtype=torch.int32, device="cuda")
    shifts = torch.arange(0, 32, bits, device="cuda", dtype=torch.int32)
    q = ((words[..., None] >> shifts) & (2 ** bits - 1)).reshape(n, k // g, g).float()
    for s, z in ((scale, zero), (scale.half(), zero.half())):
        out = torch.full((n, k + pad), 7.0, dtype=dtype, device="cuda")
        assert lib.bw_dequantize(words.data_ptr(), s.data_ptr(), CODE.get(s.dtype), z.data_ptr(), 3 if z.dtype is torch.int32 else 0,
                                 n, k, bits, g, out.data_ptr(), CODE[dtype], k + pad, _stream()) == 0
        expect = (s.float()[..., None] * (q - z.float()[..., None])).reshape(n, k).to(dtype)
        assert torch.equal(out[:, :k], expect)
        assert (out[:, k:] == 7.0).all()
