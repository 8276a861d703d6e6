"""Launches that carry a stage of the single track (ptx_*_carry), on both sides of the sizes where they run it along their own
workgroups: it runs once - a LayerNorm in place, of which a second run would show - and their own results are those of the call that carries
nothing."""
import ctypes

import pytest
import torch

from protenix_amd import _lib

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16
MODES = {"bf16": (1, BF16), "amp": (2, torch.float32), "fp32": (0, torch.float32)}   # dtype code, type of the pair rows


def _randn(seed, *shape, dtype=BF16, scale=1.0):
    return (scale * torch.randn(*shape, generator=torch.Generator().manual_seed(seed))).to("cuda", dtype)


def _both(call, mode, outputs):
    """call(stage or None, stream) without and with a stage; outputs: the tensors it fills."""
    lib = _lib.load()
    code, dt = MODES[mode]
    stream = torch.cuda.current_stream().cuda_stream
    x = [3.0 + _randn(5, 50, 384, dtype=dt) for _ in range(2)]
    gamma, beta = _randn(6, 384, dtype=dt) + 2.0, _randn(7, 384, dtype=dt)
    stages = [(ctypes.c_int64 * 32)() for _ in range(2)]
    for s, t in zip(stages, x):
        _lib.check(lib.ptx_single_layernorm_stage(s, t.data_ptr(), gamma.data_ptr(), beta.data_ptr(), t.data_ptr(), 50, 384, 1e-5,
                                                  1 if dt is BF16 else 0), "stage")
    _lib.check(lib.ptx_single_stage_run(stages[0], stream), "run")
    _lib.check(call(None, stream), "alone")
    want = [t.clone() for t in outputs]
    for t in outputs:
        t.fill_(float("nan"))
    _lib.check(call(stages[1], stream), "carrying")
    assert torch.equal(x[0], x[1])
    assert all(torch.equal(a, b) for a, b in zip(outputs, want))


@pytest.mark.parametrize("mode", ["bf16", "amp"])
@pytest.mark.parametrize("n,carries", [(93, True), (101, False), (120, False), (128, False), (146, True), (147, False), (200, False)])
@pytest.mark.parametrize("pair_bias", [True, False])
def test_output_transition(n, carries, pair_bias, mode):
    lib = _lib.load()
    code, dt = MODES[mode]
    assert bool(lib.ptx_triattn_output_transition_carries(n)) == carries
    stream = torch.cuda.current_stream().cuda_stream
    w_g, w_o = _randn(1, 128, 128, scale=0.1), _randn(2, 128, 128, scale=0.1)
    w_a, w_b, w_to = _randn(3, 256, 128, scale=0.1), _randn(4, 256, 128, scale=0.1), _randn(8, 128, 256, scale=0.1)
    packed = torch.empty(lib.ptx_triattn_output_transition_packed_elems(2), device="cuda", dtype=BF16)
    _lib.check(lib.ptx_triattn_output_transition_pack(*(t.data_ptr() for t in (w_g, w_o, w_a, w_b, w_to, packed)), 2, 1, stream), "pack")
    o, z = _randn(9, 4, n * n, 32), _randn(10, n, n, 128, dtype=dt)
    ones, pb_w = torch.ones(128, device="cuda", dtype=BF16), _randn(11, 16, 128, scale=0.1)
    out, bias = torch.empty_like(z), torch.zeros(16, n, n, device="cuda")
    args = [t.data_ptr() for t in (o, z)] + [ones.data_ptr(), None, packed.data_ptr(), ones.data_ptr(), None, out.data_ptr(), n, 128, 4, 1, 2,
                                             1e-5, 1e-5]
    args += [ones.data_ptr(), None, pb_w.data_ptr(), bias.data_ptr(), 16, 1] if pair_bias else [None, None, None, None, 0, 1]
    _both(lambda stage, st: lib.ptx_triattn_output_transition_carry(*args, 1e-5, code, stage, st), mode, [out, bias] if pair_bias else [out])


@pytest.mark.parametrize("mode,n,carries", [("bf16", 64, True), ("amp", 192, True), ("amp", 193, True), ("amp", 256, True), ("bf16", 257, False),
                                            ("amp", 257, False), ("fp32", 64, False), ("fp32", 250, False)])
def test_contraction(mode, n, carries):
    lib = _lib.load()
    code, _ = MODES[mode]
    dt = torch.float32 if mode == "fp32" else BF16
    assert bool(lib.ptx_trimul_contract_carries(n, code)) == carries
    a, b = (_randn(s, lib.ptx_trimul_operand_elems(n, 128), dtype=dt) for s in (1, 2))
    ldx = (n + 7) // 8 * 8
    x = torch.zeros(128, n, ldx, device="cuda", dtype=dt)
    live = x[:, :, :n]
    _both(lambda stage, st: lib.ptx_trimul_contract_carry(a.data_ptr(), b.data_ptr(), x.data_ptr(), n, ldx, 128, lib.ptx_key_pitch(n), code, stage,
                                                          st), mode, [live])


@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("mode,n,carries", [("bf16", 64, True), ("amp", 93, True), ("amp", 256, True), ("bf16", 257, False), ("amp", 257, False),
                                            ("fp32", 64, False)])
def test_attention_core(mode, n, carries, masked):
    lib = _lib.load()
    code, _ = MODES[mode]
    dt = torch.float32 if mode == "fp32" else BF16
    assert bool(lib.ptx_triattn_fwd_carries(n, code)) == carries
    q, o = _randn(1, 4, n, n, 32, dtype=dt, scale=0.2), torch.empty(4, n, n, 32, device="cuda", dtype=dt)
    k, vt = (_randn(s, lib.ptx_triattn_kv_elems(n, 4), dtype=dt) for s in (2, 3))
    tb = _randn(4, lib.ptx_triattn_bias_elems(n, 4), dtype=dt)
    mask = (torch.rand(n, n, generator=torch.Generator().manual_seed(5)) > 0.3).to("cuda", dt) if masked else None
    _both(lambda stage, st: lib.ptx_triattn_fwd_carry(q.data_ptr(), k.data_ptr(), vt.data_ptr(), None, tb.data_ptr(),
                                                      None if mask is None else mask.data_ptr(), o.data_ptr(), n, 4, 32, lib.ptx_key_pitch(n), 0, 1e9,
                                                      code, stage, st), mode, [o])


@pytest.mark.parametrize("mode", ["bf16", "amp"])
def test_no_rows(mode):
    """Every launch that takes a stage along runs it where it has no rows of its own."""
    lib = _lib.load()
    code, _ = MODES[mode]
    calls = [lambda s, st: lib.ptx_trimul_project_packed(*[None] * 7, 0, 128, 128, 0, 0, 1e-5, code, s, st),
             lambda s, st: lib.ptx_trimul_contract_carry(None, None, None, 0, 0, 128, 0, code, s, st),
             lambda s, st: lib.ptx_trimul_output_packed(None, 0, *[None] * 7, 0, 128, 128, 1, 1e-5, code, s, st),
             lambda s, st: lib.ptx_triattn_project_packed(*[None] * 9, 0, 128, 4, 0, 0, 1e-5, code, s, st),
             lambda s, st: lib.ptx_triattn_fwd_carry(*[None] * 7, 0, 4, 32, 0, 0, 1e9, code, s, st),
             lambda s, st: lib.ptx_triattn_output_packed(*[None] * 6, 0, 128, 4, 0, 1, 1e-5, code, s, st),
             lambda s, st: lib.ptx_trimul_output_trimul_project(None, 0, *[None] * 13, 0, 128, 128, 0, 1e-5, code, s, st),
             lambda s, st: lib.ptx_trimul_output_triattn_project(None, 0, *[None] * 14, 0, 128, 128, 4, 0, 1e-5, code, s, st),
             lambda s, st: lib.ptx_triattn_output_triattn_project(*[None] * 13, 0, 128, 4, 0, 1e-5, code, s, st),
             lambda s, st: lib.ptx_triattn_output_transition_carry(*[None] * 8, 0, 128, 4, 1, 2, 1e-5, 1e-5, *[None] * 4, 0, 1, 1e-5, code, s, st)]
    for call in calls:
        _both(call, mode, [])
