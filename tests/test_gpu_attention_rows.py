"""The triangle-attention core where its workgroups change: two rows per wave from 272 tokens on, if there are enough of them, eight
waves from 1057 on, if the queries fill them and the keys whole tiles; odd numbers of rows and of query blocks, last key tiles of one
key to a whole tile; and logits that leave the range of the reference 0, which take rows off the common path."""
import math

import pytest
import torch

from protenix_amd import _lib


def _core(n, heads, scale, g, n_keys=None):
    """q, K, V^T, bias in the core's layouts from random plain tensors, and the plain tensors."""
    lib = _lib.load()
    q, k, v = (torch.randn(heads, n, n, 32, generator=g).bfloat16() for _ in range(3))
    b = (scale * torch.randn(heads, n, n, generator=g)).bfloat16()
    pitch = lib.ptx_key_pitch(n)
    tiles, qb = pitch // 64, (n + 31) // 32
    j = torch.arange(n)
    gg, u, r = (j % 64) // 32, (j % 32) // 16, j % 16
    kd = torch.full((heads, n, tiles, 2, 2, 2, 32, 8), float("nan")).bfloat16()      # u, kk, lane half, MFMA row, d
    kd[:, :, j // 64, u, :, :, 8 * (r // 4) + 4 * gg + r % 4] = k.view(heads, n, n, 2, 2, 8).permute(2, 0, 1, 3, 4, 5)
    vd = torch.full((heads, n, tiles, 2, 2, 2, 32, 8), float("nan")).bfloat16()      # u, key group, lane half, d, key
    vd[:, :, j // 64, u, r // 8, gg, :, j % 8] = v.permute(2, 0, 1, 3)
    bd = torch.zeros(heads, qb, tiles, 2, 2, 2, 32, 8).bfloat16()
    qi = torch.arange(n)[:, None].expand(n, n)
    jj = j[None, :].expand(n, n)
    bd[:, qi // 32, jj // 64, (jj % 32) // 16, (jj % 16) // 8, (jj % 64) // 32, qi % 32, jj % 8] = b
    return (q, kd, vd, bd), (q, k, v, b), pitch


def _reference(q, k, v, b, rows, n_keys):
    # the core works in log2 units: probabilities 2^(q.k + b)
    s = torch.einsum("hiqd,hikd->hiqk", q[:, rows].float(), k[:, rows].float()) + b[:, None].float()
    p = torch.softmax(s[..., :n_keys] * math.log(2.0), dim=-1)
    return torch.einsum("hiqk,hikd->hiqd", p, v[:, rows, :n_keys].float())


@pytest.mark.gpu
@pytest.mark.parametrize("n", [33, 271, 272, 273, 351, 352, 353, 385, 417, 1057, 1152, 1280])
@pytest.mark.parametrize("scale", [1.0, 40.0])
def test_core(n, scale):
    lib, heads = _lib.load(), 2 if 256 < n < 300 else 1        # (1024 workgroups of one row and 128 queries, for two rows per wave)
    g = torch.Generator().manual_seed(n)
    dev, plain, pitch = _core(n, heads, scale, g)
    dq, dk, dv, db = (t.cuda() for t in dev)
    st = torch.cuda.current_stream().cuda_stream
    for row0, count, n_keys in ((0, n, n), (2, n - 3, n - 1), (1, n - 2, n)):
        o = torch.full((heads, n, n, 32), 7.0, dtype=torch.bfloat16, device="cuda")
        rc = lib.ptx_triattn_fwd_rows(dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), None, db.data_ptr(), None, o.data_ptr(), n, heads, 32,
                                      pitch, 0, 1e9, row0, count, n_keys, 1, st)
        assert rc == 0
        o = o.cpu()
        rows = sorted({row0, row0 + 1, row0 + count // 2, row0 + count - 2, row0 + count - 1})
        # (probabilities and outputs are rounded to 8 significant bits: 2^-8 each of a weighted mean of |v| < 5)
        err = (o[:, rows].float() - _reference(*plain, rows, n_keys)).abs().max().item()
        assert err <= 2 * 2.0 ** -8 * plain[2].abs().max().item(), (n, scale, row0, err)
        outside = [r for r in range(n) if not row0 <= r < row0 + count]
        assert bool((o[:, outside] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("rows,s,heads,with_b1", [(1, 1, 1, True), (3, 31, 4, True), (2, 64, 2, False), (5, 65, 4, True), (4, 100, 3, False),
                                                  (3, 352, 4, False), (2, 353, 4, False), (5, 385, 4, True), (2, 500, 1, True),
                                                  (2, 1057, 2, False), (1, 2056, 1, True)])
def test_standard_layouts_equal_the_repacked_operands(rows, s, heads, with_b1):
    """16-bit operands read as they are, and repacked where the output would overwrite V: the same products, bit for bit."""
    lib = _lib.load()
    g = torch.Generator().manual_seed(rows * s)
    q, k, v = (torch.randn(rows, s, heads, 32, generator=g).bfloat16().cuda() for _ in range(3))
    b2 = torch.randn(heads, s, s, generator=g).bfloat16().cuda()
    b1 = (-1e9 * (torch.rand(rows, s, generator=g) > 0.8).float()).bfloat16().cuda() if with_b1 else None
    ws = torch.empty(lib.ptx_triattn_core_workspace_elems(rows, s, heads), dtype=torch.bfloat16, device="cuda")
    st = torch.cuda.current_stream().cuda_stream
    outs = []
    for o in (torch.empty_like(v), v.clone()):
        lse = torch.empty(rows, s, heads, device="cuda")
        src = v if not outs else o
        rc = lib.ptx_triattn_core_fwd(q.data_ptr(), k.data_ptr(), src.data_ptr(), None if b1 is None else b1.data_ptr(), b2.data_ptr(),
                                      o.data_ptr(), lse.data_ptr(), ws.fill_(float("nan")).data_ptr(), 1, rows, s, heads, 32, 1, st)
        assert rc == 0
        outs.append((o, lse))
    assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
    assert bool(torch.isfinite(outs[0][0]).all())
