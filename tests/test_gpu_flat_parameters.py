"""Parameters that are views into one flat buffer, at addresses no vector load takes: what the stand-alone
LayerNorm of the single track accepts, the stack on the native path accepts as well."""
import pytest
import torch

import protenix_amd as P
from protenix_amd import ops
from oracle import pairformer_oracle as O
from tests.util import oracle_and_product, rel_err, tol

pytestmark = pytest.mark.gpu


def _view(t, offset):
    flat = torch.empty(t.numel() + 16, device=t.device, dtype=t.dtype)
    v = flat[offset:offset + t.numel()].view(t.shape)
    with torch.no_grad():
        v.copy_(t)
    return v


@pytest.mark.parametrize("native", [True, False])
@pytest.mark.parametrize("mode", ["fp32", "amp", "bf16"])
@pytest.mark.parametrize("name", ["attention_pair_bias.layernorm_a", "single_transition.layernorm1"])
def test_single_layernorm_parameters_at_any_address(name, mode, native, monkeypatch):
    dt = torch.bfloat16 if mode == "bf16" else torch.float32
    _, prod = oracle_and_product(O.PairformerStack, P.PairformerStack, n_blocks=2, dtype=torch.bfloat16)
    prod = prod.to(dt)
    s, z, pm = O.make_inputs(20, n_pad=3, dtype=torch.bfloat16)
    s, z, pm = s.to("cuda", dt), z.to("cuda", dt), pm.cuda()
    monkeypatch.setattr(ops, "native_enabled", native)

    def run():
        with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16, enabled=mode == "amp"):
            return prod(s, z, pm)
    s0, z0 = run()
    ln = prod.blocks[0].get_submodule(name)
    for offset, p in ((1, "weight"), (3, "bias")):
        setattr(ln, p, torch.nn.Parameter(_view(getattr(ln, p).detach(), offset)))
        assert getattr(ln, p).data_ptr() % 16
    s1, z1 = run()
    assert bool(torch.equal(z1, z0))        # (z never depends on s)
    if native:      # the same kernel on a copy
        same = bool(torch.equal(s1, s0))
        assert same
    else:
        # the stand-alone kernel reads such parameters element by element and sums a row of 384 in another
        # order: some sqrt(384) * 2^-24 = 1e-6 of a LayerNorm's output; in bf16 one of its roundings may move
        assert rel_err(s1, s0) <= tol(dt)
