"""Rows of the attention core whose keys are all masked (the padded rows of a batch, as the last rows of more than 256): the mean of V
where q.k and the bias drown in the mask, the masked path where they might not.  The reference is the same kernel over all rows
(ptx_triattn_fwd), which takes the masked path for every row (layers.py:286-291: (q.k + mask bias) + triangle bias in fp32)."""
import pytest
import torch

from protenix_amd import _lib

pytestmark = pytest.mark.gpu
BF16, HEADS, INF = 1, 4, 1e9


def _operands(n, seed, q_scale=0.2):
    """Random q, and random contents of the fragment-ordered K, V^T and bias (what lies beyond n keys counts for nothing)."""
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(seed)

    def randn(*shape):
        return torch.randn(*shape, device="cuda", generator=g)
    q = (randn(HEADS, n, n, 32) * q_scale).bfloat16()
    k = randn(lib.ptx_triattn_kv_elems(n, HEADS)).bfloat16()
    vt = randn(lib.ptx_triattn_kv_elems(n, HEADS)).bfloat16()
    tb = randn(lib.ptx_triattn_bias_elems(n, HEADS)).bfloat16()
    return q, k, vt, tb


def _both(n, nv, q, k, vt, tb, mask, transposed=0, gate=None):
    lib = _lib.load()
    st = torch.cuda.current_stream().cuda_stream
    outs = [torch.full((HEADS, n, n, 32), 7.0, device="cuda").bfloat16() for _ in range(2)]
    gp = None if gate is None else gate.data_ptr()
    args = (q.data_ptr(), k.data_ptr(), vt.data_ptr(), gp, tb.data_ptr(), mask.data_ptr())
    pitch = lib.ptx_key_pitch(n)
    _lib.check(lib.ptx_triattn_fwd(*args, outs[0].data_ptr(), n, HEADS, 32, pitch, transposed, INF, BF16, st), "fwd")
    _lib.check(lib.ptx_triattn_fwd_rows(*args, outs[1].data_ptr(), n, HEADS, 32, pitch, transposed, INF, nv, n - nv, n, BF16, st), "rows")
    assert (outs[1][:, :nv] == 7.0).all()                       # nothing outside the range is written
    return outs[0][:, nv:].float(), outs[1][:, nv:].float()


def _pair_mask(n, nv):
    m = torch.zeros(n, device="cuda")
    m[:nv] = 1
    return (m[:, None] * m[None, :]).bfloat16().contiguous()


# (the mean is one fp32 sum in another order, then one rounding to bf16)
REL = 2.0 ** -8


@pytest.mark.parametrize("transposed", [0, 1])
@pytest.mark.parametrize("n,nv", [(2, 1), (31, 30), (33, 32), (64, 40), (65, 1), (97, 90), (129, 128), (200, 199), (256, 250), (257, 250), (258, 257),
                                  (289, 256), (385, 353),
                                  (1536, 1530), (2049, 2048)])
def test_mean_of_v(n, nv, transposed):
    ops = _operands(n, n)
    whole, rows = _both(n, nv, *ops, _pair_mask(n, nv), transposed)
    assert (rows - whole).abs().max() <= REL * whole.abs().max()
    assert (rows == rows[:, :, :1]).all()                       # every query alike


@pytest.mark.parametrize("n,nv", [(64, 40), (97, 90), (257, 250), (300, 290)])
def test_rows_that_are_not_uniform_take_the_masked_path(n, nv):
    """Bit for bit what the whole launch gives: logits or biases that the mask does not swallow, a key that is not masked."""
    q, k, vt, tb = _operands(n, n + 1)
    mask = _pair_mask(n, nv)
    big = q.clone()
    big[1, nv] *= 200                                            # one (head, row): |q.k| beyond half of 1e9's last place
    whole, rows = _both(n, nv, big, k, vt, tb, mask)
    assert torch.equal(rows[1, 0], whole[1, 0])
    assert (rows - whole).abs().max() <= REL * whole.abs().max()
    for row in (n - 1, nv):                                      # the last row, or the first, has a key
        for key in (0, 3):
            open_ = mask.clone()
            open_[row, key] = 1
            whole, rows = _both(n, nv, q, k, vt, tb, open_)
            assert torch.equal(rows[:, row - nv], whole[:, row - nv])
            assert (rows - whole).abs().max() <= REL * whole.abs().max()
    for value in (1000.0, -float("inf"), float("nan")):          # a bias of head 0, block of queries 0, key 0
        odd = tb.clone()
        odd[0] = value
        whole, rows = _both(n, nv, q, k, vt, odd, mask)
        assert torch.equal(rows[0, :, :32].nan_to_num(9.0), whole[0, :, :32].nan_to_num(9.0))
        assert (rows - whole)[1:].abs().max() <= REL * whole[1:].abs().max()
    for t in (q, k):
        odd = t.clone()
        odd.view(-1)[-1 if t is q else 0] = float("nan")
        whole, rows = _both(n, nv, *((odd, k) if t is q else (q, odd)), vt, tb, mask)
        assert torch.equal(rows.isnan(), whole.isnan())


@pytest.mark.parametrize("n,nv", [(70, 60), (270, 260)])
def test_values_that_are_not_numbers_and_gates(n, nv):
    q, k, vt, tb = _operands(n, 5)
    odd = vt.clone()
    odd[: odd.numel() // 2: 40001] = float("nan")
    odd[1:: 50021] = float("inf")
    whole, rows = _both(n, nv, q, k, odd, tb, _pair_mask(n, nv))
    assert torch.equal(rows.isnan(), whole.isnan()) and torch.equal(rows.isinf(), whole.isinf())
    gate = torch.rand(HEADS, n, n, 32, device="cuda").bfloat16()
    whole, rows = _both(n, nv, q, k, vt, tb, _pair_mask(n, nv), gate=gate)
    assert torch.equal(rows, whole)                              # with a gate the masked path as it is
