"""Blocks and stacks that are not told to work in place leave z as it was, wherever it starts and however it lies, and
return another tensor; the first block then reads the caller's tensor itself."""
import pytest
import torch

import protenix_amd as P
from oracle import pairformer_oracle as O
from protenix_amd import ops
from tests.util import oracle_and_product, pad_mask

BF16 = torch.bfloat16


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["fp32", "bf16", "amp"])
@pytest.mark.parametrize("n,batch", [(21, 2), (300, 1)])
def test_z_is_left_as_it_was(mode, n, batch):
    _, prod = oracle_and_product(O.PairformerStack, P.PairformerStack, n_blocks=2, dtype=BF16)
    dt = BF16 if mode == "bf16" else torch.float32
    prod = prod.to(dt)
    g = torch.Generator().manual_seed(n)
    dense = torch.randn(batch, n, n, 128, generator=g).to("cuda", dt)
    s, m = torch.randn(batch, n, 384, generator=g).to("cuda", dt), torch.cat([pad_mask(n, 3)] * batch).cuda()
    room = torch.empty(dense.numel() + 1, device="cuda", dtype=dt)
    shifted = room[1:].view_as(dense).copy_(dense)                    # (contiguous, not at a multiple of 16 bytes)
    strided = dense.transpose(1, 2).contiguous().transpose(1, 2)

    def run(mod, z, **kw):
        with torch.no_grad(), torch.autocast("cuda", dtype=BF16, enabled=mode == "amp"):
            return mod(s, z, m, **kw)
    for mod in (prod, prod.blocks[0]):
        want = run(mod, dense.clone(), inplace_safe=True)
        for z in (dense, shifted, strided):
            for native in (True, False):
                ops.native_enabled = native
                try:
                    got = run(mod, z)
                finally:
                    ops.native_enabled = True
                assert torch.equal(z, strided) and got[1].data_ptr() != z.data_ptr()
                assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
