"""The operands of the triangle multiplication's product: K from n to the pitch is written as zeros, whatever lay there, by the
projection on packed weights and by the output stage that projects for the update behind it."""
import pytest
import torch

from protenix_amd import _lib

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16
MODES = {"bf16": (1, BF16, BF16), "amp": (2, torch.float32, BF16), "fp32": (0, torch.float32, torch.float32)}   # code, rows, arithmetic


def _randn(seed, *shape, dtype=BF16, scale=1.0):
    return (scale * torch.randn(*shape, generator=torch.Generator().manual_seed(seed))).to("cuda", dtype)


def _rows(t, n, c):
    """[c][n][pitch] of a tensor in the product's operand order."""
    pitch = _lib.load().ptx_key_pitch(n)
    t = t.view(c, (n + 31) // 32, pitch // 16, 2, 32, 8)
    return t.permute(0, 1, 4, 2, 3, 5).reshape(c, -1, pitch)[:, :n]


@pytest.mark.parametrize("mode,c_z", [("bf16", 128), ("amp", 128), ("fp32", 128), ("amp", 64), ("amp", 256)])
@pytest.mark.parametrize("n", [1, 20, 33, 65, 93, 96, 129, 160, 193, 230, 257, 330])
def test_projections_write_zeros_up_to_the_pitch(mode, c_z, n):
    lib = _lib.load()
    code, rows, dt = MODES[mode]
    hidden, stream = max(c_z, 128), torch.cuda.current_stream().cuda_stream
    ws = [_randn(i, hidden, c_z, dtype=dt, scale=0.1) for i in range(4)] + [_randn(5, c_z, hidden, dtype=dt), _randn(6, c_z, c_z, dtype=dt)]
    packed = torch.empty(lib.ptx_trimul_packed_elems(c_z, hidden, code), device="cuda", dtype=dt)
    _lib.check(lib.ptx_trimul_pack(*(w.data_ptr() for w in ws), packed.data_ptr(), c_z, hidden, code, stream), "pack")
    z, pitch = _randn(7, n, n, c_z, dtype=rows), lib.ptx_key_pitch(n)
    elems = lib.ptx_trimul_operand_elems(n, hidden)

    def operands():
        return [torch.full((elems,), float("nan"), device="cuda", dtype=dt) for _ in range(2)]
    for incoming in (0, 1):
        ab = operands()
        _lib.check(lib.ptx_trimul_project_packed(z.data_ptr(), None, None, None, packed.data_ptr(), ab[0].data_ptr(), ab[1].data_ptr(), n, c_z,
                                                 hidden, pitch, incoming, 1e-5, code, None, stream), "project")
        for t in ab:
            t = _rows(t, n, hidden)
            assert torch.isfinite(t).all() and (t[:, :, n:] == 0).all() and (t[:, :, :n] != 0).any()
    if mode == "fp32" or c_z == 256:
        return
    ldx, ab, out = (n + 7) // 8 * 8, operands(), torch.empty_like(z)
    x = _randn(8, hidden, n, ldx, dtype=dt)
    _lib.check(lib.ptx_trimul_output_trimul_project(x.data_ptr(), ldx, z.data_ptr(), None, None, None, None, None, packed.data_ptr(), out.data_ptr(),
                                                    None, None, packed.data_ptr(), ab[0].data_ptr(), ab[1].data_ptr(), n, c_z, hidden, pitch, 1e-5,
                                                    code, None, stream), "output and projection")
    for t in ab:
        t = _rows(t, n, hidden)
        assert torch.isfinite(t).all() and (t[:, :, n:] == 0).all() and (t[:, :, :n] != 0).any()
