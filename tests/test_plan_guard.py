"""What a plan of the native host path stands for: the package's own modules, each running its own forward.  The
record itself is examined on the CPU; on the GPU a replaced sub-module, a sub-class, a `forward` set on an
instance and a hook have to take effect, alone and in a stack."""
import types

import pytest
import torch

import protenix_amd as P
from protenix_amd import native
from oracle import pairformer_oracle as O
from tests.util import oracle_and_product, rel_err

PARTS = ["tri_mul_out", "tri_mul_in", "tri_att_start", "tri_att_end", "pair_transition", "attention_pair_bias",
         "single_transition", "single_transition.layernorm1", "tri_att_end.mha.linear_o"]


def _sub_class(m):
    m.__class__ = type("Other", (type(m),), {"forward": lambda self, x, *a, **k: x})


def _instance(m):
    m.forward = types.MethodType(lambda self, x, *a, **k: x, m)


def _hook(m):
    m.register_forward_hook(lambda *_: None)


@pytest.mark.parametrize("change", [_sub_class, _instance, _hook])
@pytest.mark.parametrize("part", PARTS)
def test_the_record_notices_another_forward(part, change):
    blk = P.PairformerBlock(c_s=64, n_heads=2).eval()
    guard = native._guard(blk)
    assert guard is not None and guard.valid() and native.runs_own_forward(blk.get_submodule(part))
    change(blk.get_submodule(part))
    assert not guard.valid() and native._guard(blk) is None
    assert not native.runs_own_forward(blk.get_submodule(part))


def test_the_record_refuses_other_classes():
    blk = P.PairformerBlock(c_s=64, n_heads=2).eval()
    guard = native._guard(blk)
    blk.tri_mul_in = torch.nn.Identity()
    assert not guard.valid() and native._guard(blk) is None
    class Mine(P.PairformerBlock):
        pass
    assert native._guard(Mine(c_s=64, n_heads=2)) is None


def test_a_forward_put_into_a_class_is_noticed(monkeypatch):
    blk = P.PairformerBlock(c_s=64, n_heads=2).eval()
    assert native.runs_own_forward(blk.tri_att_end)
    monkeypatch.setattr(P.TriangleAttention, "forward", lambda self, x, *a, **k: x)
    assert not native.runs_own_forward(blk.tri_att_end)


# For each part of a block: the weight whose zeros make its update vanish, and a forward without an update
ZEROS = {"tri_mul_out": ("linear_z", None), "tri_mul_in": ("linear_z", None), "tri_att_start": ("mha.linear_o", 0),
         "tri_att_end": ("mha.linear_o", 0), "pair_transition": ("linear_no_bias", 0),
         "attention_pair_bias": ("attention.linear_o", 0), "single_transition": ("linear_no_bias", 0)}


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["instance", "sub_class", "replaced", "patched"])
@pytest.mark.parametrize("part", list(ZEROS))
def test_another_forward_takes_effect(part, how, monkeypatch):
    """The first block of a stack (and the block alone) with one part that does nothing: as with that part's last
    weight zero."""
    weight, zero = ZEROS[part]
    _, prod = oracle_and_product(O.PairformerStack, P.PairformerStack, n_blocks=2)
    _, want_of = oracle_and_product(O.PairformerStack, P.PairformerStack, n_blocks=2)
    with torch.no_grad():
        for b in want_of.blocks[:2 if how == "patched" else 1]:     # (a class changes for every block)
            for m in ([b.get_submodule(part)] if how != "patched" else [x for x in b.modules() if type(x) is type(b.get_submodule(part))]):
                m.get_submodule(weight).weight.zero_()
    s, z, pm = (t.cuda() for t in O.make_inputs(24, n_pad=3))
    with torch.no_grad():
        prod(s, z, pm)             # (plans of the unchanged stack exist)

    def nothing(self, x, *a, **k):
        r = k.get("_residual_out")
        return r if r is not None else x + 0 if k.get("_residual_new") else x if zero is None else torch.zeros_like(x)
    blk = prod.blocks[0]
    m = blk.get_submodule(part)
    if how == "instance":
        m.forward = types.MethodType(nothing, m)
    elif how == "sub_class":
        m.__class__ = type("Other", (type(m),), {"forward": nothing})
    elif how == "replaced":
        setattr(blk, part, type("Other", (torch.nn.Module,), {"forward": nothing})())
    else:
        monkeypatch.setattr(type(m), "forward", nothing)
    for mod, ref in ((prod, want_of), (prod.blocks[0], want_of.blocks[0])):
        with torch.no_grad():
            s1, z1 = mod(s, z, pm)
            s2, z2 = ref(s, z, pm) if how != "patched" else _unpatched(monkeypatch, lambda: ref(s, z, pm), type(m), nothing)
        # (fp32 sums in another order where a stage runs in a kernel of its own)
        assert rel_err(z1, z2.cpu()) <= 1e-5 and rel_err(s1, s2.cpu()) <= 1e-5


def _unpatched(monkeypatch, f, cls, patch):
    monkeypatch.undo()
    out = f()
    monkeypatch.setattr(cls, "forward", patch)
    return out
