"""The native host path (csrc/host.cpp) against the Python path it stands in for: the same kernels in the
same order, so whole stacks, updates, LayerNorm and the attention operator are compared bit for bit,
with their gradients, and a plan notices every change of what it was made from."""
import pytest
import torch

import protenix_amd as P
from protenix_amd import native, ops
from protenix_amd.layer_norm import FusedLayerNorm
from protenix_amd.tri_attention import TriAttentionFunction
from oracle import pairformer_oracle as O
from tests.util import oracle_and_product, pad_mask

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def both(f):
    """f() on the native path, which it must have taken, and on the Python path."""
    calls = []
    real = native.host()

    class Spy:
        def __getattr__(self, name):
            calls.append(name)
            return getattr(real, name)
    native._host = Spy()
    try:
        a = f()
    finally:
        native._host = real
    assert calls
    ops.native_enabled = False
    try:
        return a, f()
    finally:
        ops.native_enabled = True


@pytest.mark.parametrize("mode,n,batch,pad,kw", [
    ("amp", 40, None, None, {}), ("amp", 33, 2, 5, {}), ("bf16", 37, None, 4, {}), ("fp32", 24, None, 3, {}),
    ("amp", 31, None, -1, {}), ("amp", 29, None, 2, dict(c_z=64, c_s=0)), ("bf16", 21, None, 2, dict(c_z=256, hidden_scale_up=True))])
def test_stack_and_block_equal_the_python_path(mode, n, batch, pad, kw):
    _, prod = oracle_and_product(O.PairformerStack, P.PairformerStack, n_blocks=4, dtype=BF16, **kw)
    dt = BF16 if mode == "bf16" else torch.float32
    prod = prod.to(dt)
    lead = () if batch is None else (batch,)
    g = torch.Generator().manual_seed(n)
    c_z, c_s = kw.get("c_z", 128), kw.get("c_s", 384)
    z = torch.randn(*lead, n, n, c_z, generator=g).to("cuda", dt)
    s = torch.randn(*lead, n, c_s, generator=g).to("cuda", dt) if c_s else None
    m = None
    if pad is not None:     # -1: an arbitrary mask
        m = torch.cat([pad_mask(n, pad)] * (batch or 1)) if pad >= 0 else (torch.rand(1, n, n, generator=g) > 0.3).float()
        m = (m if batch else m[0]).cuda()

    def run(mod):
        with torch.no_grad(), torch.autocast("cuda", dtype=BF16, enabled=mode == "amp"):
            return mod(s, z, m)
    for mod in (prod, prod.blocks[0]):
        (s1, z1), (s2, z2) = both(lambda: run(mod))
        assert torch.equal(z1, z2) and (s1 is s2 if s is None else torch.equal(s1, s2))


def test_a_plan_notices_changes():
    _, prod = oracle_and_product(O.PairformerStack, P.PairformerStack, n_blocks=2, dtype=BF16)
    s, z, m = (t.cuda() for t in O.make_inputs(19, n_pad=2))

    def same():
        with torch.no_grad():
            (s1, z1), (s2, z2) = both(lambda: prod(s, z, m))
        assert torch.equal(z1, z2) and torch.equal(s1, s2)
        return z1
    last = same()
    blk = prod.blocks[1]
    changes = [lambda: blk.tri_mul_in.linear_g.weight.add_(0.1),
               lambda: setattr(blk.tri_att_end.linear, "weight", torch.nn.Parameter(blk.tri_att_end.linear.weight * 2)),
               lambda: setattr(blk, "pair_transition", prod.blocks[0].pair_transition),
               lambda: prod.blocks.append(prod.blocks[0]), lambda: setattr(blk.tri_att_start, "inf", 2.0)]
    for change in changes:
        with torch.no_grad():
            change()
        now = same()
        assert not torch.equal(now, last)
        last = now
    # hooks below a block leave it to the Python path
    seen = []
    prod.blocks[0].single_transition.register_forward_pre_hook(lambda *_: seen.append(1))
    with torch.no_grad():
        _, z1 = prod(s, z, m)
    assert seen and torch.equal(z1, last)


@pytest.mark.parametrize("scale,offset", [(True, True), (True, False), (False, True), (False, False)])
def test_layer_norm_and_gradients(scale, offset):
    ln = FusedLayerNorm(48, create_scale=scale, create_offset=offset).cuda()
    for frozen in ((), ("weight",), ("bias",)):
        for name, p in ln.named_parameters():
            p.requires_grad_(name not in frozen)
        x = torch.randn(5, 7, 48, device="cuda")

        def run():
            xx = x.clone().requires_grad_()
            y = ln(xx)
            wrt = [xx, *(p for p in ln.parameters() if p.requires_grad)]
            return (y.detach(), *torch.autograd.grad((y * x).sum(), wrt))
        a, b = both(run)
        assert all(torch.equal(u, v) for u, v in zip(a, b))


@pytest.mark.parametrize("bias1", [True, False])
@pytest.mark.parametrize("b2_grad", [True, False])
def test_attention_operator_and_gradients(bias1, b2_grad):
    q, k, v = (torch.randn(2, 3, 33, 4, 32, device="cuda", dtype=BF16) for _ in range(3))
    b1 = torch.randn(2, 3, 1, 1, 33, device="cuda", dtype=BF16) if bias1 else None
    b2 = torch.randn(1, 1, 4, 33, 33, device="cuda")       # (another type, broadcast over the batch)

    def run():
        ts = [t.clone().requires_grad_() for t in (q, k, v)] + [b2.clone().requires_grad_(b2_grad)]
        o = TriAttentionFunction.apply(*ts[:3], b1, ts[3])
        return (o.detach(), *torch.autograd.grad((o * q).sum(), [t for t in ts if t.requires_grad]))
    a, b = both(run)
    assert all(torch.equal(u, w) and u.dtype == w.dtype for u, w in zip(a, b))
