"""Backward of the fused attention operator (ptx_triattn_core_bwd behind
TriAttentionFunction): dQ, dK, dV and dBias2 against torch autograd through the oracle's
softmax_attention (the reference's torch-path _attention, layers.py:276-296) on the same
operands; the contract is the reference's TriAttentionFunction.backward
(tri_attention/op.py:79-163).  Rows whose every key is masked are left out of the operands: their
log-sum-exp is about -1.4e9, where fp32 no longer resolves log2 of the key count, so the
reference's M format itself carries no usable gradient for them."""
import math

import pytest
import torch

import protenix_amd as P
from oracle import pairformer_oracle as O
from tests.util import rel_err, tol

pytestmark = pytest.mark.gpu
DTYPES = [torch.float32, torch.bfloat16]


def _operands(B, N, S, H, dtype, seed, n_masked=0, b2_batch=None):
    g = torch.Generator().manual_seed(seed)
    q = (torch.randn(B, N, S, H, 32, generator=g) / math.sqrt(32)).to(dtype)
    k = torch.randn(B, N, S, H, 32, generator=g).to(dtype)
    v = torch.randn(B, N, S, H, 32, generator=g).to(dtype)
    do = torch.randn(B, N, S, H, 32, generator=g).to(dtype)
    mask = torch.ones(B, N, S)
    if n_masked:
        mask[..., S - n_masked:] = 0
        mask[:, 1] = (torch.rand(B, S, generator=g) > 0.5).float()
        mask[:, 1, 0] = 1                          # never a row with every key masked
    b1 = (1e9 * (mask - 1)).reshape(B, N, 1, 1, S).to(dtype)
    b2 = torch.randn(B if b2_batch is None else b2_batch, 1, H, S, S, generator=g).to(dtype)
    return q, k, v, b1, b2, do


def _autograd_reference(q, k, v, b1, b2, do):
    q, k, v, b2 = (t.float().clone().requires_grad_(True) for t in (q, k, v, b2))
    o = O.softmax_attention(q.transpose(-2, -3), k.transpose(-2, -3), v.transpose(-2, -3),
                            [b1.float(), b2]).transpose(-2, -3)
    o.backward(do.float())
    return o.detach(), q.grad, k.grad, v.grad, b2.grad


def _product(q, k, v, b1, b2, do, grad_b2=True):
    q, k, v, b2 = (t.cuda().requires_grad_(r) for t, r in ((q, True), (k, True), (v, True), (b2, grad_b2)))
    o = P.TriAttentionFunction.apply(q, k, v, b1.cuda(), b2)
    o.backward(do.cuda())
    return o.detach(), q.grad, k.grad, v.grad, b2.grad


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("B,N,S,H,n_masked", [(1, 32, 32, 4, 0), (1, 64, 64, 4, 0), (2, 37, 37, 4, 5),
                                              (1, 8, 100, 2, 7), (1, 130, 130, 2, 0), (1, 3, 200, 8, 16)])
def test_gradients_against_autograd_of_the_torch_path(dtype, B, N, S, H, n_masked):
    ops = _operands(B, N, S, H, dtype, seed=N * 11 + S, n_masked=n_masked)
    want = _autograd_reference(*ops)
    got = _product(*ops)
    for name, g, w in zip(("O", "dQ", "dK", "dV", "dBias2"), got, want):
        assert g.shape == w.shape and g.dtype == dtype, name
        # dBias2 sums N rows of bf16-rounded products: allow the rounding of the sum itself
        assert rel_err(g, w) <= tol(dtype), name


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("N,S", [(5, 96), (3, 50)])
def test_no_bias1_is_a_bias1_of_zeros(dtype, N, S):
    """Without a mask bias the kernels read a row of Bias2 in its place and weigh it with zero:
    same gradients as with a Bias1 of zeros, and as the torch path's."""
    q, k, v, b1, b2, do = _operands(1, N, S, 2, dtype, seed=S)
    want = _autograd_reference(q, k, v, b1, b2, do)
    with_zeros = _product(q, k, v, b1, b2, do)
    qc, kc, vc, b2c = (t.cuda().requires_grad_(True) for t in (q, k, v, b2))
    P.TriAttentionFunction.apply(qc, kc, vc, None, b2c).backward(do.cuda())
    for name, g, z, w in zip(("dQ", "dK", "dV", "dBias2"), (qc.grad, kc.grad, vc.grad, b2c.grad),
                             with_zeros[1:], want[1:]):
        assert torch.equal(g, z), name
        assert rel_err(g, w) <= tol(dtype), name


@pytest.mark.parametrize("dtype", DTYPES)
def test_bias2_broadcast_over_the_batch_and_not_requiring_grad(dtype):
    ops = _operands(2, 16, 40, 4, dtype, seed=9, n_masked=3, b2_batch=1)
    want = _autograd_reference(*ops)
    got = _product(*ops)
    assert got[4].shape == ops[4].shape
    for g, w in zip(got, want):
        assert rel_err(g, w) <= tol(dtype)
    skipped = _product(*ops, grad_b2=False)
    assert skipped[4] is None
    for a, b in zip(skipped[:4], got[:4]):
        assert torch.equal(a, b)


def test_caller_level_function_differentiates():
    """layers.py:539-583 spelling: q, k, v [*, H, Q, C], the result [*, Q, H, C]."""
    g = torch.Generator().manual_seed(2)
    S, H = 48, 4
    q = (torch.randn(S, H, S, 32, generator=g) / math.sqrt(32))
    k, v = torch.randn(S, H, S, 32, generator=g), torch.randn(S, H, S, 32, generator=g)
    b1 = torch.zeros(S, 1, 1, S)
    b2 = torch.randn(1, H, S, S, generator=g)
    do = torch.randn(S, S, H, 32, generator=g)
    ref = [t.clone().requires_grad_(True) for t in (q, k, v, b2)]
    O.softmax_attention(ref[0], ref[1], ref[2], [b1, ref[3]]).transpose(-2, -3).backward(do)
    dev = [t.cuda().requires_grad_(True) for t in (q, k, v, b2)]
    P.tri_attention(dev[0], dev[1], dev[2], [b1.cuda(), dev[3]]).backward(do.cuda())
    for a, b in zip(dev, ref):
        assert a.grad.shape == b.grad.shape
        assert rel_err(a.grad, b.grad) <= 1e-4


def test_bias1_requiring_grad_is_refused():
    q, k, v, b1, b2, _ = _operands(1, 4, 32, 2, torch.float32, seed=1)
    with pytest.raises(RuntimeError, match="Bias1"):
        P.TriAttentionFunction.apply(q.cuda(), k.cuda(), v.cuda(), b1.cuda().requires_grad_(True), b2.cuda())


@pytest.mark.parametrize("dtype", DTYPES)
def test_full_size_invariants(dtype):
    """N = S = 768, 4 heads (the benchmark's attention shape), where autograd on the CPU is out
    of reach: (1) dS sums to zero over the keys of every (row, query, head), so dBias2 summed
    over keys is the rounding noise of 768 rows; (2) the operator is linear in dO; (3) a
    64-row slice agrees with autograd on the CPU."""
    N = S = 768
    q, k, v, b1, b2, do = _operands(1, N, S, 4, dtype, seed=77, n_masked=40)
    _, dq, dk, dv, db2 = _product(q, k, v, b1, b2, do)
    scale = db2.float().abs().max().item()
    assert db2.float().sum(-1).abs().max().item() <= (5e-4 if dtype == torch.float32 else 1.0) * scale
    _, dq2, dk2, dv2, db22 = _product(q, k, v, b1, b2, (2 * do.float()).to(dtype))
    for a, b in ((dq, dq2), (dk, dk2), (dv, dv2), (db2, db22)):
        assert rel_err(2 * a.float(), b.float()) <= (1e-5 if dtype == torch.float32 else 1e-2)
    sl = slice(100, 164)
    want = _autograd_reference(q[:, sl], k[:, sl], v[:, sl], b1[:, sl], b2, do[:, sl])
    for g, w in zip((dq, dk, dv), want[1:4]):
        assert rel_err(g[:, sl], w) <= tol(dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("N,S,H", [(15, 64, 1), (16, 64, 1), (65, 33, 3), (131, 72, 2), (300, 65, 1)])
def test_sliced_dbias2_equals_one_slice(dtype, N, S, H):
    """dBias2's rows in one walk (no scratch given) and in slices whose sums are added: 2 (from 16 rows on) to 32
    slices of unequal length, sizes off the vector lengths.  Two fp32 sums of N terms in another
    order differ by at most N 2^-24 of the sum of magnitudes, here below 2e-4 of the largest element; then one
    rounding to the output type.  The other outputs do not depend on it."""
    from protenix_amd import _lib
    lib = _lib.load()
    n_parts = lib.ptx_triattn_core_bwd_partial_elems(N, S, H)
    assert (n_parts == 0) == (N < 16) and n_parts % (H * S * S) == 0
    q, k, v, b1, b2, do = (t.cuda() for t in _operands(1, N, S, H, dtype, seed=N))
    o, lse = P.tri_attention_forward(q, k, v, b1, b2, return_lse=True)

    def run(parts):
        outs = [torch.full_like(t, float("nan")) for t in (q, k, v, b2)]
        delta = torch.empty(N * S * H, device="cuda")
        _lib.check(lib.ptx_triattn_core_bwd_sliced(
            *(t.data_ptr() for t in (q, k, v, b1, b2, o, lse, do, *outs, delta)), parts, 1, N, S, H, 32,
            {torch.float32: 0, torch.bfloat16: 1}[dtype], torch.cuda.current_stream().cuda_stream), "bwd")
        return outs
    one = run(None)
    parts = torch.full((n_parts + 64,), float("nan"), device="cuda")
    sliced = run(parts.data_ptr())
    assert torch.isnan(parts[n_parts:]).all()            # nothing beyond the scratch that was asked for
    assert all(torch.equal(a, b) for a, b in zip(one[:3], sliced[:3]))
    assert rel_err(sliced[3], one[3]) <= (2e-4 if dtype == torch.float32 else 2e-4 + 2.0 ** -8)


@pytest.mark.parametrize("N,S,H", [(2, 7, 1), (3, 8, 1), (5, 9, 3), (3, 31, 2), (2, 32, 4), (9, 33, 1), (2, 127, 2), (2, 128, 1), (2, 129, 3),
                                   (3, 255, 1), (2, 256, 2), (2, 257, 1), (2, 383, 2), (3, 384, 1), (64, 385, 3), (47, 391, 4),
                                   (48, 511, 4), (64, 512, 3), (48, 513, 4), (192, 767, 1), (48, 768, 4), (48, 769, 4),
                                   (33, 129, 4), (43, 255, 3), (65, 256, 2), (32, 256, 4), (48, 257, 4), (86, 264, 4), (48, 383, 4), (86, 384, 4),
                                   (129, 384, 4), (54, 513, 4), (54, 640, 4)])
def test_whole_rows_at_a_time(N, S, H):
    """16-bit rows of every class of the backward that takes a (row, head) at a time and of its neighbours that do not, in length and in
    number: a vector more and less than a block, the last keys' shifted Bias2 vectors, dQ over one to eight waves.  One row has
    a Bias1 of -inf for half of its keys, and Bias2 has -inf at one key for one query; the weight there is 0.  The reference is
    autograd in fp32 on the same device."""
    low = -math.inf
    q, k, v, b1, b2, do = _operands(1, N, S, H, torch.bfloat16, seed=N + S, n_masked=min(3, S - 2))
    b1[:, 0, ..., S // 2:] = low
    b2[..., S - 2, 1] = low
    _, dq, dk, dv, db2 = _product(q, k, v, b1, b2, do)
    want = _autograd_reference(*(t.cuda() for t in (q, k, v, b1, b2, do)))
    for name, g, w in zip(("dQ", "dK", "dV", "dBias2"), (dq, dk, dv, db2), want[1:]):
        assert torch.isfinite(g).all() and rel_err(g, w) <= tol(torch.bfloat16), name
    assert (dk[:, 0, S // 2:] == 0).all() and (dv[:, 0, S // 2:] == 0).all() and (db2[..., S - 2, 1] == 0).all()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("with_bias1", [True, False])
@pytest.mark.parametrize("N,S,H", [(3, 40, 2), (2, 7, 1), (3, 200, 1), (2, 385, 1), (2, 770, 1)])
def test_bias2_of_minus_infinity_has_weight_zero(dtype, with_bias1, N, S, H):
    """In every kernel of the backward, as in the forward: finite gradients, those of the torch path, and none for that logit."""
    q, k, v, b1, b2, do = _operands(1, N, S, H, dtype, seed=S)
    b2[..., S - 2, 1] = -math.inf
    b2[..., 0, S // 2:] = -math.inf
    want = _autograd_reference(q, k, v, b1, b2, do)
    qc, kc, vc, b2c = (t.cuda().requires_grad_(True) for t in (q, k, v, b2))
    P.TriAttentionFunction.apply(qc, kc, vc, b1.cuda() if with_bias1 else None, b2c).backward(do.cuda())
    for name, g, w in zip(("dQ", "dK", "dV", "dBias2"), (qc.grad, kc.grad, vc.grad, b2c.grad), want[1:]):
        assert torch.isfinite(g).all() and rel_err(g, w) <= tol(dtype), name
    assert (b2c.grad[..., S - 2, 1] == 0).all() and (b2c.grad[..., 0, S // 2:] == 0).all()


@pytest.mark.parametrize("N,S,H", [(17, 33, 1), (24, 97, 4), (40, 160, 4), (16, 191, 2),       # two waves of one block
                                   (64, 192, 4), (70, 193, 5), (33, 257, 8), (64, 288, 4),      # three waves of two blocks
                                   (64, 224, 4), (65, 289, 4), (64, 321, 5), (17, 800, 4),      # four waves of two blocks
                                   # few rows, one slice: spans of tiles per XCD, each form, and tiles in turn (513)
                                   (5, 97, 4), (3, 300, 2), (7, 520, 4), (5, 600, 4), (3, 1100, 4), (3, 513, 4), (2, 1030, 1)])
def test_dbias2_in_workgroups_of_every_size(N, S, H):
    """The three forms of dBias2's walk, at sizes that fill their tiles, just pass them and fall short of them, masked keys among
    them.  Tolerance as for the other gradients: the reference's O and log-sum-exp are not rounded."""
    q, k, v, b1, b2, do = (t.cuda() for t in _operands(1, N, S, H, torch.bfloat16, seed=N * S, n_masked=min(9, S // 3)))
    want = _autograd_reference(q, k, v, b1, b2, do)[4]
    got = _product(q, k, v, b1, b2, do)[4]
    assert torch.isfinite(got).all()
    assert rel_err(got, want) <= tol(torch.bfloat16)
