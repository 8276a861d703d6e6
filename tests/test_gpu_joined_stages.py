"""Output stages that project for the update behind them (csrc/pairproj.hip, pp_joined) and products that carry a stage of the
single track: the native path, which joins them, against the Python path, which launches every stage by itself - the same
arithmetic, so bit for bit - on both sides of the sizes at which the joined launches, their tiles and the carrying
products change, odd sizes and padded masks included."""
import pytest
import torch

import protenix_amd as P
from oracle import pairformer_oracle as O
from tests.test_gpu_native_host import both
from tests.util import oracle_and_product, pad_mask

BF16 = torch.bfloat16


@pytest.mark.gpu
@pytest.mark.parametrize("mode,c_z,n,batch,pad", [
    ("amp", 128, 1, 1, 0), ("amp", 128, 7, 2, 1), ("bf16", 128, 31, 2, 0), ("amp", 128, 93, 1, 6), ("amp", 128, 101, 1, 0), ("amp", 128, 102, 1, 0), ("bf16", 128, 128, 1, 3), ("amp", 128, 128, 2, 0), ("amp", 128, 146, 1, 0),
    ("amp", 128, 147, 1, 0), ("bf16", 64, 255, 1, 3), ("amp", 64, 256, 1, 0), ("bf16", 128, 9, 1, 0), ("amp", 128, 159, 1, 3), ("bf16", 128, 160, 1, 0),
    ("amp", 128, 161, 1, 5), ("amp", 128, 193, 1, 0), ("amp", 128, 256, 1, 9), ("amp", 128, 257, 1, 0), ("bf16", 128, 355, 1, 0),
    ("bf16", 128, 479, 1, 0), ("bf16", 128, 484, 1, 0), ("amp", 128, 527, 1, 17), ("amp", 128, 528, 1, 0), ("amp", 128, 596, 1, 0),
    ("amp", 128, 601, 1, 4), ("amp", 64, 5, 2, 1), ("bf16", 64, 158, 1, 0), ("amp", 64, 165, 1, 2), ("amp", 64, 396, 1, 0),
    ("amp", 256, 9, 1, 1), ("amp", 256, 97, 1, 0), ("bf16", 256, 203, 1, 3), ("amp", 256, 256, 1, 0), ("amp", 256, 257, 1, 0)])
def test_joined_equal_separate(mode, c_z, n, batch, pad):
    kw = {128: {}, 64: dict(c_z=64, c_s=0, num_intermediate_factor=2), 256: dict(c_z=256, hidden_scale_up=True)}[c_z]
    _, prod = oracle_and_product(O.PairformerStack, P.PairformerStack, n_blocks=3, dtype=BF16, **kw)
    dt = BF16 if mode == "bf16" else torch.float32
    prod = prod.to(dt)
    g = torch.Generator().manual_seed(n)
    z = torch.randn(batch, n, n, c_z, generator=g).to("cuda", dt)
    s = torch.randn(batch, n, 384, generator=g).to("cuda", dt) if c_z != 64 else None
    m = torch.cat([pad_mask(n, pad)] * batch).cuda() if pad else None

    def run():
        with torch.no_grad(), torch.autocast("cuda", dtype=BF16, enabled=mode == "amp"):
            return prod(s, z, m)
    (s1, z1), (s2, z2) = both(run)
    assert torch.equal(z1, z2) and (s1 is s2 if s is None else torch.equal(s1, s2))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [30, 129, 200])
def test_without_a_single_track(n):
    _, prod = oracle_and_product(O.PairformerStack, P.PairformerStack, n_blocks=2, dtype=BF16, c_s=0)
    z = torch.randn(1, n, n, 128, generator=torch.Generator().manual_seed(n)).cuda()
    m = (torch.rand(1, n, n, generator=torch.Generator().manual_seed(n)) > 0.3).float().cuda()

    def run():
        with torch.no_grad(), torch.autocast("cuda", dtype=BF16):
            return prod(None, z, m)
    (_, z1), (_, z2) = both(run)
    assert torch.equal(z1, z2)
