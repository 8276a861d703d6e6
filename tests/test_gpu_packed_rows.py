"""The row-local kernels on packed weights (csrc/pairproj.hip), the transition on few rows
(csrc/transition_small.hip) and the single track's stages on packed weights, at the sizes where their
dispatch changes: against the general kernels they stand in for (csrc/rowgemm.hip, attnout.hip,
transition.hip), which the oracle tests hold to the reference.

Both sides form the same products of the same rounded operands in fp32 and round at the same places, so that
they differ by the order of fp32 sums and, in 16-bit arithmetic, by the rounding of a value that such a
difference moved across a boundary: one bf16 step (2^-8) of an element, 4e-3 of the largest."""
import pytest
import torch

import protenix_amd as P
from protenix_amd import ops, triangular
from oracle import pairformer_oracle as O
from tests.util import oracle_and_product, pad_mask, rel_err

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16
TOL = {"fp32": 1e-5, "bf16": 4e-3, "amp": 4e-3}


def _call(mod, args, mode):
    with torch.no_grad(), torch.autocast("cuda", dtype=BF16, enabled=mode == "amp"):
        return mod(*args)


# (sizes around the lines of in_row_blocks / out_row_blocks, and both kinds of tiles: n a multiple of 8 or not)
SIZES = ([(128, m, n) for m in ("amp", "bf16") for n in (159, 160, 161, 319, 320, 447, 448, 449)]
         # (from 352, 480, 704 and 896 on, rows in bf16 take the kernels with all weights in LDS, out of the same packed
         # buffer; 360 has some of the four stages there, 904 all, 903 none)
         + [(128, "bf16", n) for n in (344, 352, 360, 480, 704, 903, 904)] + [(128, "amp", 704)]
         + [(128, "fp32", n) for n in (31, 33, 160, 323)]
         + [(64, m, n) for m in ("amp", "fp32") for n in (32, 161, 399, 400, 450)]
         + [(256, m, n) for m in ("amp", "bf16") for n in (33, 95, 96, 97, 199, 200, 203)])


@pytest.mark.parametrize("c_z,mode,n", SIZES)
def test_updates_equal_the_general_kernels(c_z, mode, n, monkeypatch):
    hidden, heads = (256, 8) if c_z == 256 else (128, 4)
    dt = BF16 if mode == "bf16" else torch.float32
    g = torch.Generator().manual_seed(n)
    z = torch.randn(1, n, n, c_z, generator=g).to("cuda", dt)
    mask = (torch.rand(1, n, n, generator=g) > 0.2).to("cuda", dt)
    mods = [oracle_and_product(getattr(O, c), getattr(P, c), c_z, hidden, dtype=BF16)[1]
            for c in ("TriangleMultiplicationOutgoing", "TriangleMultiplicationIncoming")]
    mods += [oracle_and_product(O.TriangleAttention, P.TriangleAttention, c_z, 32, heads, starting=s, dtype=BF16)[1]
             for s in (True, False)]
    for mod in (m.to(dt) for m in mods):
        got = _call(mod, (z, mask), mode)
        with monkeypatch.context() as m:
            m.setattr(triangular, "_with_packed", lambda w, *_: w)
            m.setattr(ops, "native_enabled", False)
            m.setattr(ops, "late_gate_enabled", c_z == 128)
            general = type(mod)(c_z, hidden) if hasattr(mod, "_outgoing") else type(mod)(c_z, 32, heads, starting=mod.starting)
            general.load_state_dict(mod.state_dict())
            want = _call(general.to("cuda", dt).eval(), (z, mask), mode)
        assert got.dtype == want.dtype and rel_err(got, want) <= TOL[mode], type(mod).__name__


@pytest.mark.parametrize("mode", ["fp32", "bf16", "amp"])
@pytest.mark.parametrize("c,factor", [(64, 2), (128, 4), (256, 4)])
def test_transition_on_few_rows_equals_the_one_on_many(c, factor, mode):
    """Rows of a call large enough for the fused kernel against the same rows in small calls: one row, a tile of 32 and
    its neighbours, and a partial last tile."""
    if c == 256 and mode == "fp32":
        pytest.skip("no fp32 arithmetic on rows of 256 channels")
    dt = BF16 if mode == "bf16" else torch.float32
    mod = oracle_and_product(O.Transition, P.Transition, c, factor, dtype=BF16)[1].to(dt)
    x = torch.randn(400 * 400, c, generator=torch.Generator().manual_seed(c)).to("cuda", dt)
    want = _call(mod, (x,), mode)
    for rows in (1, 31, 32, 33, 95, 4099):
        assert rel_err(_call(mod, (x[:rows],), mode), want[:rows]) <= TOL[mode], rows


@pytest.mark.parametrize("mode,n,kw", [("amp", 130, {}), ("amp", 257, {}), ("bf16", 200, {}), ("fp32", 150, {}), ("amp", 450, {}),
                                       ("amp", 120, dict(c_z=256, hidden_scale_up=True))])
def test_carried_single_track_equals_the_python_path(mode, n, kw):
    """Every tile size of the linear stages, weights in fragment order, riding on the pair kernels: bit for bit what
    the stages give as launches of their own on the weights as they are (the Python path)."""
    _, prod = oracle_and_product(O.PairformerStack, P.PairformerStack, n_blocks=2, dtype=BF16, **kw)
    dt = BF16 if mode == "bf16" else torch.float32
    prod = prod.to(dt)
    g = torch.Generator().manual_seed(n)
    z = torch.randn(n, n, kw.get("c_z", 128), generator=g).to("cuda", dt)
    s = torch.randn(n, 384, generator=g).to("cuda", dt)
    m = pad_mask(n, 3)[0].cuda()
    s1, z1 = _call(prod, (s, z, m), mode)
    ops.native_enabled = False
    try:
        s2, z2 = _call(prod, (s, z, m), mode)
    finally:
        ops.native_enabled = True
    assert torch.equal(z1, z2) and torch.equal(s1, s2)
