"""The two instruments of ops.py - launches timed one by one, workspaces filled with NaN - on the native host path,
which is what calls run on: a poisoned call gives the same bits, a timed one lists the launches of that path."""
import pytest
import torch

import protenix_amd as P
from protenix_amd import native, ops
from oracle import pairformer_oracle as O
from tests.util import oracle_and_product, pad_mask

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


@pytest.fixture
def native_calls(monkeypatch):
    """Names taken from the extension module."""
    names = []
    real = native.host()

    class Spy:
        def __getattr__(self, name):
            names.append(name)
            return getattr(real, name)
    monkeypatch.setattr(native, "_host", Spy())
    return names


def _stack(mode, n, pad, batch=None, **kw):
    _, prod = oracle_and_product(O.PairformerStack, P.PairformerStack, n_blocks=3, dtype=BF16, **kw)
    dt = BF16 if mode == "bf16" else torch.float32
    lead = () if batch is None else (batch,)
    g = torch.Generator().manual_seed(n)
    c_z, c_s = kw.get("c_z", 128), kw.get("c_s", 384)
    z = torch.randn(*lead, n, n, c_z, generator=g).to("cuda", dt)
    s = torch.randn(*lead, n, c_s, generator=g).to("cuda", dt) if c_s else None
    m = torch.cat([pad_mask(n, pad)] * (batch or 1)).cuda() if pad else None
    prod = prod.to(dt)

    def run():
        with torch.no_grad(), torch.autocast("cuda", dtype=BF16, enabled=mode == "amp"):
            return prod(s, z, m if batch or m is None else m[0])
    return run


@pytest.mark.parametrize("mode,n,pad,batch,kw", [
    ("amp", 40, 0, None, {}), ("amp", 33, 5, 2, {}), ("bf16", 37, 4, None, {}), ("fp32", 24, 3, None, {}), ("amp", 130, 0, None, {}),
    ("amp", 29, 2, None, dict(c_z=64, c_s=0)), ("bf16", 21, 2, None, dict(c_z=256, hidden_scale_up=True))])
def test_poisoned_workspaces_change_nothing(mode, n, pad, batch, kw, native_calls, monkeypatch):
    run = _stack(mode, n, pad, batch, **kw)
    want = run()
    del native_calls[:]
    monkeypatch.setattr(ops, "poison_workspaces", True)
    for _ in range(2):
        got = run()
        assert all(a is b if a is None else bool(torch.equal(a, b)) for a, b in zip(got, want))
    assert native_calls.count("Call") == 2


def test_the_native_workspace_is_poisoned():
    """The switch reaches the buffers of the native path: each is filled before the launches."""
    run = _stack("amp", 40, 0)
    run()
    torch.cuda.synchronize()
    ops.poison_workspaces = True
    try:
        prof = torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CPU])
        with prof:
            run()
    finally:
        ops.poison_workspaces = False
    # the pair workspace, the pair bias and the single track's scratch
    assert sum(e.count for e in prof.key_averages() if e.key == "aten::fill_") >= 3


def test_timed_launches_are_those_of_the_native_path(native_calls, monkeypatch):
    run = _stack("amp", 40, 0)
    want = run()
    del native_calls[:]
    monkeypatch.setattr(ops, "kernel_timer", {})
    got = run()
    times = ops.kernel_times(ops.kernel_timer)
    assert native_calls.count("Call") == 1
    assert all(bool(torch.equal(a, b)) for a, b in zip(got, want))
    counts = {k: len(v) for k, v in times.items()}
    # three blocks; only the last one's single track has launches of its own
    assert counts == {"trimul_project": 6, "trimul_contract": 6, "trimul_output": 6, "triattn_project": 6, "triattn_fwd": 6,
                      "triattn_output": 3, "triattn_output_transition": 3, "layernorm": 2, "linear": 3, "single_attention": 1,
                      "swiglu": 1}
    assert all(t > 0 for v in times.values() for t in v)
