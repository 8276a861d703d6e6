"""Plans made in C++ from the modules' parameters (csrc/host.cpp, csrc/params.hip): the same bits as the Python path,
which has its weights converted and packed by torch and the pack entry points, whatever type, place, order and
address the parameters come in."""
import ctypes

import pytest
import torch

import protenix_amd as P
from protenix_amd import _lib, native, ops
from oracle import pairformer_oracle as O
from tests.test_gpu_native_host import both
from tests.util import oracle_and_product, pad_mask

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16
CODE = {torch.float32: _lib.PTX_F32, BF16: _lib.PTX_BF16}


def _pack(items):
    class Item(ctypes.Structure):
        _fields_ = [("src", ctypes.c_void_p), ("dst", ctypes.c_void_p), ("rows", ctypes.c_int64), ("cols", ctypes.c_int),
                    ("src_dtype", ctypes.c_int), ("dst_dtype", ctypes.c_int), ("fragments", ctypes.c_int)]
    a = (Item * len(items))(*(Item(s.data_ptr(), d.data_ptr(), r, c, CODE[s.dtype], CODE[d.dtype], int(f)) for s, d, r, c, f in items))
    _lib.check(_lib.load().ptx_param_pack(ctypes.addressof(a), len(items), torch.cuda.current_stream().cuda_stream), "param_pack")


def test_param_pack():
    """Every pair of types, plain and in fragment order, sizes around a workgroup's share, more items than a launch
    takes; unaligned sources; values torch rounds to even, subnormals, infinities."""
    items, want = [], []
    for src_t in (torch.float32, BF16):
        for dst_t in (torch.float32, BF16):
            for rows, cols in [(1, 1), (1, 7), (3, 683), (1, 2048), (1, 2049), (16, 384), (0, 5)] * 3:
                x = torch.randn(rows * cols + 1, device="cuda").to(src_t)[1:].view(rows, cols)
                if cols == 683:
                    x.view(-1)[:8] = torch.tensor([1 + 2**-8, 1 + 3 * 2**-8, 2.0**-130, -2.0**-149, float("inf"), -float("inf"), 3.4e38,
                                                   0.0]).to(src_t)
                items.append((x, torch.full((rows, cols), -7.0, device="cuda", dtype=dst_t), rows, cols, False))
                want.append(x.to(dst_t))
            for rows, cols in [(16, 32), (32, 96), (384, 384), (48, 1536)]:
                x = torch.randn(rows, cols, device="cuda").to(src_t)
                ve = 16 // torch.empty((), dtype=dst_t).element_size()
                items.append((x, torch.full((rows * cols,), -7.0, device="cuda", dtype=dst_t), rows, cols, True))
                want.append(x.to(dst_t).view(rows // 16, 16, cols // 32, 8 // ve, 4, ve).permute(0, 2, 3, 4, 1, 5).reshape(-1))
    _pack(items)
    for (_, got, *_), w in zip(items, want):
        assert bool(torch.equal(got, w))


def test_param_pack_refusals():
    x, y = torch.zeros(15, 32, device="cuda"), torch.zeros(480, device="cuda")
    for rows, cols, dt in ((15, 32, 0), (16, 24, 0), (16, 32, 3)):
        with pytest.raises(RuntimeError, match="param_pack"):
            class Item(ctypes.Structure):
                _fields_ = [("src", ctypes.c_void_p), ("dst", ctypes.c_void_p), ("rows", ctypes.c_int64), ("v", ctypes.c_int * 4)]
            it = Item(x.data_ptr(), y.data_ptr(), rows, (ctypes.c_int * 4)(cols, dt, dt, 1))
            _lib.check(_lib.load().ptx_param_pack(ctypes.addressof(it), 1, None), "")


def _native(f):
    calls = []
    real = native.host()

    class Spy:
        def __getattr__(self, name):
            calls.append(name)
            return getattr(real, name)
    native._host = Spy()
    try:
        return f()
    finally:
        native._host = real
        assert "Call" in calls


def _changed(prod, how):
    """The stack with its parameters in another type, place, order or at another address."""
    for m in prod.modules():
        for name, p in list(m.named_parameters(recurse=False)):
            t = p.detach()
            if how == "transposed" and t.dim() == 2:
                t = t.t().contiguous().t()
            elif how == "flat":
                buf = torch.empty(t.numel() + 3, device=t.device, dtype=t.dtype)
                buf[3:].view(t.shape).copy_(t)
                t = buf[3:].view(t.shape)
            elif how == "cpu":
                t = t.cpu()
            elif how == "bf16":
                t = t.to(BF16)
            elif how == "mixed" and t.dim() == 2:
                t = t.to(BF16)
            elif how == "double":
                t = t.double()
            setattr(m, name, torch.nn.Parameter(t, requires_grad=False))
    return prod


@pytest.mark.parametrize("how", ["transposed", "flat", "cpu", "bf16", "mixed", "double"])
@pytest.mark.parametrize("mode,kw", [("amp", {}), ("fp32", {}), ("amp", dict(c_z=64, c_s=0)), ("amp", dict(c_z=256, hidden_scale_up=True))])
def test_stack_with_parameters_of_any_kind(mode, kw, how):
    _, prod = oracle_and_product(O.PairformerStack, P.PairformerStack, n_blocks=2, dtype=BF16, **kw)
    prod = prod.float()             # (values that bf16 holds: the same in every type)
    n, c_z, c_s = 25, kw.get("c_z", 128), kw.get("c_s", 384)
    g = torch.Generator().manual_seed(3)
    z = torch.randn(1, n, n, c_z, generator=g).cuda()
    s = torch.randn(1, n, c_s, generator=g).cuda() if c_s else None

    def run():
        with torch.no_grad(), torch.autocast("cuda", dtype=BF16, enabled=mode == "amp"):
            return prod(s, z, pad_mask(n, 4).cuda())
    (s1, z1), (s2, z2) = both(run)
    assert bool(torch.equal(z1, z2)) and (s is None or bool(torch.equal(s1, s2)))
    _changed(prod, how)
    (s1, z1) = _native(run)
    assert bool(torch.equal(z1, z2)) and (s is None or bool(torch.equal(s1, s2)))


@pytest.mark.parametrize("mode", ["amp", "bf16", "fp32"])
@pytest.mark.parametrize("how", ["as they are", "transposed", "cpu"])
@pytest.mark.parametrize("cls,args", [(P.TriangleMultiplicationIncoming, (128, 128)), (P.TriangleMultiplicationOutgoing, (64, 128)),
                                      (P.TriangleAttention, (128, 32, 4)), (P.TriangleAttentionEndingNode, (64, 32, 4))])
def test_updates(cls, args, how, mode):
    dt = BF16 if mode == "bf16" else torch.float32
    m = _changed(O.seed_parameters_(cls(*args)).to("cuda", dt).eval(), how)
    z = torch.randn(1, 23, 23, args[0], device="cuda").to(dt)

    def run():
        with torch.no_grad(), torch.autocast("cuda", dtype=BF16, enabled=mode == "amp"):
            return (m(z, pad_mask(23, 3).cuda()),)
    (a,), (b,) = both(run)
    assert bool(torch.equal(a, b))


def test_a_plan_keeps_no_copies_beside_its_own():
    """The native path neither fills the modules' own caches nor keeps what it converted on the way."""
    _, prod = oracle_and_product(O.PairformerBlock, P.PairformerBlock, dtype=BF16)
    prod = prod.float()
    z, s = torch.randn(1, 16, 16, 128, device="cuda"), torch.randn(1, 16, 384, device="cuda")

    def run():
        with torch.no_grad(), torch.autocast("cuda", dtype=BF16):
            return prod(s, z, None)
    run()
    native._plans.clear()
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    out = run()
    del out
    torch.cuda.synchronize()
    kept = torch.cuda.memory_allocated() - before
    lib = _lib.load()
    pair = 2 * (2 * lib.ptx_trimul_packed_elems(128, 128, 1) + 2 * lib.ptx_triattn_packed_elems(128, 4, 1)
                + lib.ptx_triattn_output_transition_packed_elems(4))
    single = 4 * 384 * 384 * (4 + 1 + 3 * 4)
    assert pair + single <= kept <= pair + single + 64 * 1024      # (vectors; the allocator's rounding)
    assert all(m._cache._key is None for m in prod.modules() if hasattr(m, "_cache"))


def test_weights_of_another_shape_are_left_to_the_python_path():
    _, prod = oracle_and_product(O.PairformerBlock, P.PairformerBlock)
    prod.tri_mul_out.linear_z.weight = torch.nn.Parameter(torch.zeros(64, 128, device="cuda"))
    z = torch.randn(1, 16, 16, 128, device="cuda")
    with torch.no_grad():
        assert native._block_plan(prod, z, torch.float32, torch.float32) is None


@pytest.mark.parametrize("at", [0, 1, 2, 3])
@pytest.mark.parametrize("how", ["hook", "other", "another class"])
def test_a_block_without_a_plan_leaves_the_rest_to_python(at, how):
    """The blocks before it have run natively by then, on the caller's z and s."""
    _, prod = oracle_and_product(O.PairformerStack, P.PairformerStack, n_blocks=4)
    s, z, pm = (t.cuda() for t in O.make_inputs(21, n_pad=2))
    with torch.no_grad():
        want = prod(s, z, pm)
        seen = []
        blk = prod.blocks[at]
        if how == "hook":
            blk.tri_mul_in.register_forward_hook(lambda *_: seen.append(1))
        elif how == "another class":
            class Wrapped(torch.nn.Module):
                def __init__(self, blk):
                    super().__init__()
                    self.inner = blk

                def forward(self, *a, **k):
                    seen.append(1)
                    return self.inner(*a, **k)
            prod.blocks[at] = Wrapped(blk).eval()
        else:
            fwd = blk.forward
            blk.forward = lambda *a, **k: (seen.append(1), fwd(*a, **k))[1]
        for _ in range(2):
            got = prod(s, z, pm)
            assert all(bool(torch.equal(a, b)) for a, b in zip(got, want))
    assert len(seen) == 2


def test_blocks_of_growing_size_in_one_stack():
    """Two heads' worth of single track first, then more: the scratch of a call grows while stages wait."""
    _, a = oracle_and_product(O.PairformerStack, P.PairformerStack, n_blocks=3)
    a.blocks[1].single_transition = O.seed_parameters_(P.Transition(384, 8)).cuda().eval()
    s, z, pm = (t.cuda() for t in O.make_inputs(40, n_pad=2))

    def run():
        with torch.no_grad():
            return a(s, z, pm)
    got = _native(run)              # (new weights: block by block)
    again = _native(run)            # (kept plans: all at once)
    (s1, z1), (s2, z2) = both(run)
    for x, y in ((got[0], s2), (again[0], s2), (s1, s2), (got[1], z2), (again[1], z2), (z1, z2)):
        assert bool(torch.equal(x, y))
