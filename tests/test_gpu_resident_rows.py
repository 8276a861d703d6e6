"""Where a projection takes the kernel that keeps all weights in LDS out of the packed buffer (csrc/pairproj.hip,
pp_resident), also on fp32 rows: against the general kernels on weights as they are, and, in a stack, the stages of the
single track that such a projection cannot carry against the Python path, bit for bit."""
import pytest
import torch

import protenix_amd as P
from protenix_amd import _lib, ops, triangular
from oracle import pairformer_oracle as O
from tests.util import oracle_and_product

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def _call(mod, args, mode):
    with torch.no_grad(), torch.autocast("cuda", dtype=BF16, enabled=mode == "amp"):
        return mod(*args)


def test_the_lines():
    lib = _lib.load()

    def takes(stage, dtype, *ns):
        return [bool(lib.ptx_row_stage_resident(stage, n, 128, 128, dtype)) for n in ns]
    for stage, first in enumerate((704, 480, 352, 896)):
        assert takes(stage, _lib.PTX_BF16, first - 8, first, first + 1, first + 8, 8192) == [False, True, False, True, True]
    assert takes(2, _lib.PTX_MIXED, 472, 480, 484, 1784, 1792) == [False, True, False, True, False]
    assert takes(0, _lib.PTX_MIXED, 2040, 2048, 2049) == [False, True, False]
    assert takes(1, _lib.PTX_MIXED, 768, 2048) == takes(3, _lib.PTX_MIXED, 768, 2048) == [False, False]
    for stage in range(4):
        assert takes(stage, _lib.PTX_F32, 768, 2048) == [False, False]
        assert not lib.ptx_row_stage_resident(stage, 768, 64, 128, _lib.PTX_BF16)


@pytest.mark.parametrize("kind,n", [("att", 472), ("att", 480), ("att", 488), ("att", 1784), ("mul", 2048)])
def test_fp32_rows_equal_the_general_kernels(kind, n, monkeypatch):
    mods = ([oracle_and_product(O.TriangleAttention, P.TriangleAttention, 128, 32, 4, starting=s, dtype=BF16)[1] for s in (True, False)]
            if kind == "att" else [oracle_and_product(getattr(O, c), getattr(P, c), 128, 128, dtype=BF16)[1]
                                   for c in ("TriangleMultiplicationOutgoing", "TriangleMultiplicationIncoming")])
    z = torch.randn(1, n, n, 128, device="cuda", generator=torch.Generator("cuda").manual_seed(n))
    for mod in (m.float() for m in mods):
        got = _call(mod, (z, None), "amp").float()
        with monkeypatch.context() as m:
            m.setattr(triangular, "_with_packed", lambda w, *_: w)
            m.setattr(ops, "native_enabled", False)
            mod._cache._key = None
            want = _call(mod, (z, None), "amp").float()
        mod._cache._key = None
        # (the same rounded operands, fp32 sums in another order, one bf16 step of an element at most: see
        # tests/test_gpu_packed_rows.py)
        assert ((got - want).abs().max() / want.abs().max()).item() <= 4e-3


@pytest.mark.parametrize("mode,n", [("amp", 472), ("amp", 480), ("amp", 520), ("amp", 2048), ("bf16", 352), ("bf16", 480), ("bf16", 704)])
def test_stages_that_do_not_ride(mode, n):
    _, prod = oracle_and_product(O.PairformerStack, P.PairformerStack, n_blocks=3 if n < 1000 else 2, dtype=BF16)
    dt = BF16 if mode == "bf16" else torch.float32
    prod = prod.to(dt)
    g = torch.Generator("cuda").manual_seed(n)
    z = torch.randn(n, n, 128, generator=g, device="cuda").to(dt)
    s = torch.randn(n, 384, generator=g, device="cuda").to(dt)
    s1, z1 = _call(prod, (s, z, None), mode)
    ops.native_enabled = False
    try:
        s2, z2 = _call(prod, (s, z, None), mode)
    finally:
        ops.native_enabled = True
    assert bool(torch.equal(z1, z2)) and bool(torch.equal(s1, s2))
