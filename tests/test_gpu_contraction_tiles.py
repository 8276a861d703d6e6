"""The triangle product at the sizes where its kernels and their tiles change: below, at and above every tile edge, channel
counts the XCDs do not share evenly, rows at vectors and not; rows past n hold NaN, K past n zeros, as the projection leaves them."""
import ctypes

import pytest
import torch

from protenix_amd import _lib


def _operand(m, n, pitch, dtype):
    """[c, n, n] in the contraction's fragment order: (row block, K step, half-wave, row, 8 K values)."""
    c, rb, ks = m.shape[0], (n + 31) // 32, pitch // 16
    full = torch.full((c, rb * 32, ks * 16), float("nan"), dtype=dtype)
    full[:, :n] = 0
    full[:, :n, :n] = m
    return full.view(c, rb, 32, ks, 2, 8).permute(0, 1, 3, 4, 2, 5).contiguous().cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("n,c", [(1, 8), (31, 3), (32, 8), (33, 9), (64, 8), (65, 8), (93, 11), (128, 8), (129, 8), (192, 8), (193, 8),
                                 (216, 3), (255, 8), (257, 9), (320, 8), (384, 3), (385, 8), (431, 3), (513, 3), (577, 3), (640, 9)])
def test_every_tile_edge(n, c, dtype):
    lib = _lib.load()
    g = torch.Generator().manual_seed(n)
    a, b = (torch.randn(c, n, n, generator=g).to(dtype) for _ in range(2))
    pitch = lib.ptx_key_pitch(n)
    fa, fb = _operand(a, n, pitch, dtype), _operand(b, n, pitch, dtype)
    ref = a.double() @ b.double().transpose(1, 2)
    # fp32 sums of n terms, rounded once to the result's type (unit roundoff 2^-24; bf16, of 8 significant bits, 2^-8)
    bound = 2.0 ** (-24 if dtype == torch.float32 else -8) * ref.abs() + 1.01 * n * 2.0 ** -24 * (a.double().abs() @ b.double().abs().transpose(1, 2))
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for ldx in sorted({n, (n + 7) // 8 * 8}):
        x = torch.full((c, n, ldx), 7.0, device="cuda", dtype=dtype)
        rc = lib.ptx_trimul_contract_ld(fa.data_ptr(), fb.data_ptr(), x.data_ptr(), n, ldx, c, pitch, 0 if dtype == torch.float32 else 1, stream)
        assert rc == 0
        y = x.cpu().double()[:, :, :n]
        assert bool(((y - ref).abs() <= bound).all()), (n, c, ldx)
