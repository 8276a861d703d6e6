"""The triangle-attention core's common path takes every probability against the softmax reference 0.  It is entered where that is
the reference of every row's first half tile (the largest logit within 14 of 0, 2^20.2), looks at its sums at the end, and waves
with one beyond 1e12 = 2^39.9 start again: logits on either side of both lines, early and late; key ranges of less than a tile, one
tile, and one key more; rows whose bits are their own affair."""

import pytest
import torch

import protenix_amd as P
from oracle import pairformer_oracle as O
from protenix_amd import _lib
from tests.util import rel_err, tol
from test_gpu_attention_rows import _core, _reference, test_standard_layouts_equal_the_repacked_operands as _standard_layouts


def _add(dev_bias, plain_bias, queries, keys, value):
    """Bias of every one of the queries at every one of the keys, in the core's layout and in the plain one."""
    qi, j = (t.reshape(-1) for t in torch.meshgrid(torch.as_tensor(queries), torch.as_tensor(keys), indexing="ij"))
    plain_bias[:, qi, j] += value
    dev_bias[:, qi // 32, j // 64, (j % 32) // 16, (j % 16) // 8, (j % 64) // 32, qi % 32, j % 8] = plain_bias[:, qi, j]


@pytest.mark.gpu
@pytest.mark.parametrize("n", [65, 130, 353, 1280])
@pytest.mark.parametrize("where", ["first", "last", "all"])
# log2 units: see above (2^128 and more: infinity)
@pytest.mark.parametrize("value", [18.0, 22.0, 30.0, 38.0, 42.0, 60.0, 100.0, 200.0, -100.0])
def test_logits_away_from_zero(n, where, value):
    lib, heads = _lib.load(), 1
    g = torch.Generator().manual_seed(n)
    (q, kd, vd, bd), (pq, pk, pv, pb), pitch = _core(n, heads, 1.0, g)
    keys = range(n) if where == "all" else [5 if where == "first" else n - 1]
    _add(bd, pb, range(n) if n < 200 else [37, 38], keys, value)
    dq, dk, dv, db = (t.cuda() for t in (q, kd, vd, bd))
    st = torch.cuda.current_stream().cuda_stream
    o = torch.full((heads, n, n, 32), 7.0, dtype=torch.bfloat16, device="cuda")
    assert lib.ptx_triattn_fwd(dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), None, db.data_ptr(), None, o.data_ptr(), n, heads, 32,
                               pitch, 0, 1e9, 1, st) == 0
    o = o.cpu()
    rows = [0, 1, n // 2, n - 2, n - 1]
    # (probabilities and outputs are rounded to 8 significant bits: 2^-8 each of a weighted mean of |v| < 5)
    err = (o[:, rows].float() - _reference(pq, pk, pv, pb, rows, n)).abs().max().item()
    assert err <= 2 * 2.0 ** -8 * pv.abs().max().item(), (n, where, value, err)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [130, 353, 1280])
@pytest.mark.parametrize("n_keys", [1, 16, 17, 63, 64, 65, 128, 129])
def test_few_keys(n, n_keys):
    lib, heads = _lib.load(), 1
    g = torch.Generator().manual_seed(n_keys)
    dev, plain, pitch = _core(n, heads, 1.0, g)
    dq, dk, dv, db = (t.cuda() for t in dev)
    st = torch.cuda.current_stream().cuda_stream
    o = torch.full((heads, n, n, 32), 7.0, dtype=torch.bfloat16, device="cuda")
    assert lib.ptx_triattn_fwd_rows(dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), None, db.data_ptr(), None, o.data_ptr(), n, heads, 32,
                                    pitch, 0, 1e9, 0, n, n_keys, 1, st) == 0
    rows = [0, 1, n // 2, n - 1]
    err = (o.cpu()[:, rows].float() - _reference(*plain, rows, n_keys)).abs().max().item()
    assert err <= 2 * 2.0 ** -8 * plain[2].abs().max().item(), (n, n_keys, err)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [65, 200, 353])
@pytest.mark.parametrize("key", [0, 63, 64, 130, 199, 352])
@pytest.mark.parametrize("value", [0.0, 60.0, 100.0])
def test_up_to_a_masked_key(n, key, value):
    """A row leaves the common path where its first masked key is; logits as above, at a key before it and in the last tile."""
    if key >= n:
        pytest.skip("no such key")
    lib, heads = _lib.load(), 1
    g = torch.Generator().manual_seed(n)
    (q, kd, vd, bd), (pq, pk, pv, pb), pitch = _core(n, heads, 1.0, g)
    _add(bd, pb, [37, 38], [5], value)
    _add(bd, pb, [40], [n - 1 if n - 1 != key else n - 2], value)
    mask = torch.ones(n, n).bfloat16()
    mask[:, key] = 0
    mask[1] = 1                                   # a row without masked keys
    mask[2, key:] = 0                             # (key = 0: all of them)
    mask[2, 0] = 1
    dq, dk, dv, db, dm = (t.cuda() for t in (q, kd, vd, bd, mask))
    st = torch.cuda.current_stream().cuda_stream
    o = torch.full((heads, n, n, 32), 7.0, dtype=torch.bfloat16, device="cuda")
    assert lib.ptx_triattn_fwd(dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), None, db.data_ptr(), dm.data_ptr(), o.data_ptr(), n, heads, 32,
                               pitch, 0, 1e9, 1, st) == 0
    o = o.cpu()
    for row in (0, 1, 2, n - 1):
        keys = mask[row].bool()
        ref = _reference(pq, pk[:, :, keys], pv[:, :, keys], pb[:, :, keys], [row], int(keys.sum()))
        # (as above; the masked path adds ln 2 * (q.k) and the bias in fp32: 1e-6 of a logit of 100)
        err = (o[:, [row]].float() - ref).abs().max().item()
        assert err <= 2 * 2.0 ** -8 * pv.abs().max().item(), (n, key, value, row, err)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,s", [(3, 353), (2, 640), (1, 1535), (1, 1536), (2, 1536), (21, 1600), (2, 2049)])
def test_operator_without_bias1(rows, s):
    """Up to 1535 positions, and beyond where the rows are few (up to 512 workgroups of 128 queries; 21 of 1600 are more, and
    repacked in both calls), the operator's operands are read as they are."""
    _standard_layouts(rows, s, 2, False)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,s", [(3, 353), (1, 1535), (2, 1536), (21, 1600)])
def test_operator_without_bias1_against_full_precision(rows, s):
    """On both sides of those lines, against the oracle on the same operands in fp32."""
    g = torch.Generator().manual_seed(s)
    q, k, v = (torch.randn(1, rows, s, 2, 32, generator=g).bfloat16() for _ in range(3))
    q, b2 = (q.float() / 32 ** 0.5).bfloat16(), torch.randn(1, 1, 2, s, s, generator=g).bfloat16()
    got = P.TriAttentionFunction.apply(*(t.cuda() for t in (q, k, v)), None, b2.cuda()).float().cpu()
    want = O.softmax_attention(*(t.float().transpose(-2, -3) for t in (q, k, v)), [b2.float()]).transpose(-2, -3)
    assert rel_err(got, want) <= tol(torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [40, 65, 130, 353])
@pytest.mark.parametrize("cut", [16, 32, 64, 128])
def test_first_keys_at_minus_infinity(n, cut):
    """A bias of -inf has weight zero also where a query has no other key in its first half tile, or first tiles."""
    if cut >= n:
        pytest.skip("no key left")
    lib, heads = _lib.load(), 1
    g = torch.Generator().manual_seed(n)
    (q, kd, vd, bd), (pq, pk, pv, pb), pitch = _core(n, heads, 1.0, g)
    _add(bd, pb, [0, 3, 37], range(cut), -float("inf"))
    _add(bd, pb, [5], [j for j in range(n) if j % 32 < 16], -float("inf"))       # the first half of every tile
    dq, dk, dv, db = (t.cuda() for t in (q, kd, vd, bd))
    st = torch.cuda.current_stream().cuda_stream
    o = torch.full((heads, n, n, 32), 7.0, dtype=torch.bfloat16, device="cuda")
    assert lib.ptx_triattn_fwd(dq.data_ptr(), dk.data_ptr(), dv.data_ptr(), None, db.data_ptr(), None, o.data_ptr(), n, heads, 32,
                               pitch, 0, 1e9, 1, st) == 0
    rows = [0, n // 2, n - 1]
    # (as above; the reference's softmax gives such keys weight zero)
    err = (o.cpu()[:, rows].float() - _reference(pq, pk, pv, pb, rows, n)).abs()
    assert bool((err <= 2 * 2.0 ** -8 * pv.abs().max()).all()), (n, cut, err.max().item())


@pytest.mark.gpu
@pytest.mark.parametrize("s", [40, 200])
def test_first_keys_at_minus_infinity_in_full_precision(s):
    g = torch.Generator().manual_seed(s)
    q, k, v = (torch.randn(1, 3, s, 2, 32, generator=g) for _ in range(3))
    b1, b2 = torch.zeros(1, 3, 1, 1, s), torch.randn(1, 1, 2, s, s, generator=g)
    q = q / 32 ** 0.5
    b2[..., 3, torch.arange(s) % 32 < 16] = -float("inf")        # the first half of every tile
    got = P.TriAttentionFunction.apply(*(t.cuda() for t in (q, k, v, b1, b2))).cpu()
    want = O.softmax_attention(*(t.transpose(-2, -3) for t in (q, k, v)), [b1, b2]).transpose(-2, -3)
    assert rel_err(got, want) <= tol(torch.float32)


def _rows(lib, dev, n, heads, pitch, row0, count, n_keys=None, o=None):
    o = torch.full((heads, n, n, 32), 7.0, dtype=torch.bfloat16, device="cuda") if o is None else o
    q, k, v, b = dev
    assert lib.ptx_triattn_fwd_rows(q.data_ptr(), k.data_ptr(), v.data_ptr(), None, b.data_ptr(), None, o.data_ptr(), n, heads, 32, pitch,
                                    0, 1e9, row0, count, n_keys or n, 1, torch.cuda.current_stream().cuda_stream) == 0
    return o


@pytest.mark.gpu
@pytest.mark.parametrize("n", [130, 271, 272, 273, 353, 1152, 1280])
@pytest.mark.parametrize("q_scale", [0.5, 1.0, 2.0, 4.0])
def test_a_row_has_the_same_bits_in_any_company(n, q_scale):
    """Rows by themselves and in a launch of all, whose workgroups take one or two of them, four or eight waves: logits that leave
    the reference 0 in the first half tile of some rows, in later tiles of others, and rows that never do."""
    lib, heads = _lib.load(), 2 if 256 < n < 340 else 1        # (enough rows for two per wave)
    g = torch.Generator().manual_seed(n)
    (q, kd, vd, bd), (pq, pk, pv, pb), pitch = _core(n, heads, 1.0, g)
    q = q.float()
    q[:, ::3] *= q_scale
    q[:, 1::5] *= 0.25
    _add(bd, pb, [37], [n - 1], 45.0)                      # (log2 units) beyond the limit in the last tile
    _add(bd, pb, [70], [64], 120.0)
    dev = [t.cuda() for t in (q.bfloat16(), kd, vd, bd)]
    whole = _rows(lib, dev, n, heads, pitch, 0, n)
    assert bool(torch.isfinite(whole).all())
    for row in sorted({0, 1, 2, 3, n // 2, n // 2 + 1, n - 2, n - 1}):
        assert torch.equal(_rows(lib, dev, n, heads, pitch, row, 1)[:, row], whole[:, row]), (n, row)
    pairs_the_other_way = _rows(lib, dev, n, heads, pitch, 1, n - 1)
    assert torch.equal(pairs_the_other_way[:, 1:], whole[:, 1:])


@pytest.mark.gpu
@pytest.mark.parametrize("n", [272, 353, 1280])
def test_rows_behind_the_range_do_not_matter(n):
    """An odd number of rows: the last one's partner in a workgroup of two lies behind the range, whatever is there."""
    lib, heads = _lib.load(), 2 if 256 < n < 340 else 1        # (enough rows for two per wave)
    g = torch.Generator().manual_seed(n)
    dev, _, pitch = _core(n, heads, 1.0, g)
    dev = [t.cuda() for t in dev]
    dev[0] = dev[0] * 4                                    # (logits whose sums depend on the reference they are taken against)
    count = n - 30 + n % 2 - 1
    assert count % 2 == 1
    want = _rows(lib, dev, n, heads, pitch, 0, count)
    for what in (float("nan"), 3.0e38, 50.0):
        other = [t.clone() for t in dev]
        other[0][:, count:] = what
        got = _rows(lib, other, n, heads, pitch, 0, count)
        assert torch.equal(got[:, :count], want[:, :count]) and bool((got[:, count:] == 7.0).all()), what


@pytest.mark.gpu
@pytest.mark.parametrize("n", [64, 130, 300, 1280])
def test_the_largest_probability_is_exact_at_large_logits(n):
    """From logits of 14 on the reference is the first half tile's maximum, whose probability is 1.  Two keys, at 2^24.125 and
    2^22.5 (q = 0, so the logits are the bias): against the reference 0 the first would be rounded by 3.0e-3 of itself, the second by
    1e-4; against the first, the second's 2^-1.625 is rounded by 1e-4.  What is left is the outputs' rounding, 2^-9 at most of
    each and, over n 32 of them, some 1e-4 on average."""
    lib, heads = _lib.load(), 1
    g = torch.Generator().manual_seed(n)
    (q, kd, vd, bd), (_, _, pv, pb), pitch = _core(n, heads, 0.0, g)
    _add(bd, pb, range(n), range(n), -60.0)
    for key, steps in ((5, (84.0, 0.125)), (9, (82.0, 0.5))):       # (each sum is a bf16 number)
        for step in steps:
            _add(bd, pb, range(n), [key], step)
    vd[:, :, 0, 0, 0, 0, :, 5] = 0                         # V of key 5 is 0: half 0, key group 0, lane half 0
    dev = [t.cuda() for t in (torch.zeros_like(q), kd, vd, bd)]
    o = _rows(lib, dev, n, heads, pitch, 0, n).cpu().double()
    v9 = pv[:, :, 9].double()                              # [head][row][channel]
    ratio = (o / v9[:, :, None]).mean().item()
    want = 1.0 / (1.0 + 2.0 ** 1.625)
    assert abs(ratio / want - 1.0) <= 5e-4, ratio / want - 1.0
