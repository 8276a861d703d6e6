"""Python's side of the native host path (csrc/host.cpp): which calls it takes, and the plans - weights
laid out for the kernels, with a record of the parameters they came from - it takes them with.

Plans live here, keyed weakly by module: they are built on a module's first call, checked on every call
(a replaced or modified parameter, a replaced sub-module, another class, a replaced `forward` or a
registered hook makes a plan stale) and go away with the module.  A plan stands for this package's own
classes only, each running its own `forward`.  What the native path does not cover is refused here
(run_blocks says how many blocks it ran, run_update returns False) and runs through the Python path, which has the same kernels
in the same order and all the error messages.
"""
from __future__ import annotations

import weakref
from typing import Optional

import torch
import torch.nn.modules.module as _nn_module

from . import ops

_plans: "weakref.WeakKeyDictionary" = weakref.WeakKeyDictionary()
_host = None
# plain attributes of the modules that the plans depend on
_ATTRS = ["inf", "no_heads", "c_hidden", "n", "n_heads", "num_heads", "c_in", "c_z", "c_s", "eps", "starting", "_outgoing",
          "precision"]


def host():
    """The extension module, built together with the kernel library."""
    global _host
    if _host is None:
        from . import _lib
        lib = _lib.load()
        try:
            from . import _host as mod
        except ImportError as e:
            raise RuntimeError("protenix_amd: the native host path (_host.so) is missing or stale; rebuild with "
                               "`python -m protenix_amd.build`") from e
        if mod.abi_version() != lib.ptx_version():
            raise RuntimeError("protenix_amd: _host.so and libprotenix_amd.so differ; rebuild with `python -m protenix_amd.build`")
        _host = mod
    return _host


_own: Optional[tuple] = None


def _own_classes() -> tuple:
    """(the classes a plan may stand for, as a set; each with the function that was its forward when this
    was first asked for)."""
    global _own
    if _own is None:
        from . import layer_norm, pairformer, primitives, transformer, triangular as tri
        classes = [layer_norm.FusedLayerNorm, primitives.Linear, primitives.Transition, tri.TriangleMultiplicativeUpdate,
                   tri.TriangleMultiplicationOutgoing, tri.TriangleMultiplicationIncoming, tri.Attention,
                   tri.TriangleAttention, tri.TriangleAttentionEndingNode, transformer.Attention,
                   transformer.AttentionPairBias, pairformer.PairformerBlock, torch.nn.Sigmoid]
        _own = (set(classes), [(c, c.forward) for c in classes])
    return _own


def runs_own_forward(module) -> bool:
    """Whether calling `module` runs the forward its class in this package has, and nothing else (no `forward` of a
    subclass, of the instance or put into the class, no hooks): its kernels may then be issued without the call."""
    return leading_own((module,)) == 1


def leading_own(modules) -> int:
    """How many of `modules`, from the first on, run their own forward (see runs_own_forward)."""
    classes, forwards = _own_classes()
    if not all(c.forward is f for c, f in forwards):
        return 0
    count = 0
    for m in modules:
        if type(m) not in classes or "forward" in m.__dict__ or m._forward_hooks or m._forward_pre_hooks:
            break
        count += 1
    return count


def _usable(z: torch.Tensor) -> bool:
    return (ops.use_native() and z.is_cuda and not torch.is_grad_enabled() and z.dim() >= 3 and z.shape[-2] == z.shape[-3]
            and z.numel() > 0 and z.dtype in (torch.float32, torch.bfloat16)
            and not _nn_module._global_forward_hooks and not _nn_module._global_forward_pre_hooks
            and all(c.forward is f for c, f in _own_classes()[1]))


def _guard(module):
    """A record of what the module's plans are made from, or None where it cannot be relied on (hooks, other
    classes, parameters without version counters)."""
    g = host().Guard(module, _ATTRS, _own_classes()[0])
    return g if g.valid() else None


def _masks(z: torch.Tensor, mask: Optional[torch.Tensor], cd: torch.dtype) -> list:
    """Per pair tensor: (mask, transposed mask, valid tokens or None) as ops.py hands them to the kernels."""
    if mask is None:
        return []
    from .triangular import _per_batch
    n = z.shape[-2]
    out = []
    for m in _per_batch(z, mask)[1]:
        nv = ops.padded_tail(m, n)
        mm = ops._mask_for(m, z, cd)
        out.append((None, None, None) if mm is None else (mm, ops._mask_for(m, z, cd, transpose=True), nv))
    return out


def _aligned(t: torch.Tensor) -> torch.Tensor:
    """t, or a copy of it where it does not start at a multiple of 16 bytes: the single track's stages read whole
    vectors, unlike the stand-alone kernels of the Python path."""
    return t if t.data_ptr() % 16 == 0 else t.clone()


def _block_plan(blk, z, cd, sd):
    """A valid plan for this block, or None."""
    key = (cd, sd if blk.c_s > 0 else None, z.device.index, z.dtype)
    plans = _plans.setdefault(blk, {})
    plan = plans.get(key)
    if plan is None or not plan.valid():
        guard = _guard(blk)
        plan = plans[key] = None if guard is None else host().make_block(guard, blk, z, cd, sd)
    return plan


def plans_of(module) -> list:
    """Every plan kept for `module` and what is below it: a recorded graph holds them, since it has their weights'
    addresses and a plan is replaced when a parameter is."""
    return [plan for m in module.modules() for plan in _plans.get(m, {}).values()]


def run_blocks(owner, blocks, s: Optional[torch.Tensor], z: torch.Tensor, pair_mask: Optional[torch.Tensor], in_place: bool):
    """The blocks on (s, z): (the new s - None without a single track -, the new z - z itself if `in_place` -, how many of the
    blocks were run).  What follows the first block without a plan is left to the caller, as is everything where the
    count is 0.  z is contiguous, and at a multiple of 16 bytes if it is not to be changed (the first block then reads it
    and writes another tensor).  `owner`: the module the list of plans is kept with."""
    if not _usable(z) or not z.is_contiguous():
        return s, z, 0
    ac = ops.autocast_compute_dtype(z)
    cd = ops.compute_dtype(z)
    if ac is not None and cd == z.dtype:
        return s, z, 0
    if pair_mask is not None and not (pair_mask.is_cuda and pair_mask.dim() >= 2):
        return s, z, 0
    single = any(b.c_s > 0 for b in blocks)
    sd = None
    if single:
        n = z.shape[-2]
        if s is None or not s.is_cuda or s.dim() < 2 or s.shape[-2] != n or s.numel() // (n * s.shape[-1]) != z.numel() // (
                n * n * z.shape[-1]) or any(b.c_s != s.shape[-1] for b in blocks):
            return s, z, 0
        sd = s.dtype
    key = ("stack", cd, sd, z.device.index, z.dtype)
    kept = _plans.setdefault(owner, {}).get(key)
    if (kept is not None and len(kept[0]) == len(blocks) and all(a() is b for a, b in zip(kept[0], blocks))
            and host().first_stale(kept[1]) < 0):
        plans = kept[1]
        call, out = _call(s, z, pair_mask, cd, single, in_place)
        call.blocks(plans)
    else:
        # a plan is made while the kernels of the blocks before it run
        plans, call = [], None
        for b in blocks:
            plan = _block_plan(b, z, cd, sd)
            if plan is None:
                break
            plans.append(plan)
            if call is None:
                call, out = _call(s, z, pair_mask, cd, single, in_place)
            call.blocks([plan])
        if call is None:
            return s, z, 0
        if len(plans) == len(blocks):
            _plans[owner][key] = ([weakref.ref(b) for b in blocks], plans)
    return call.finish(), out, len(plans)


def _call(s, z, pair_mask, cd, single, in_place):
    out = z if in_place else torch.empty_like(z)
    return host().Call(_aligned(s.contiguous()) if single else s, out, z, _masks(z, pair_mask, cd), ops.kernel_timer,
                       ops.poison_workspaces), out


def run_update(module, z: torch.Tensor, cd: torch.dtype, mask: Optional[torch.Tensor], out: torch.Tensor, add: bool,
               transposed: Optional[bool] = None) -> bool:
    """One triangle update of every pair tensor of z (contiguous) into out; False: take the Python path.
    `transposed`: None for a triangle multiplication."""
    if not _usable(z) or (mask is not None and not mask.is_cuda):
        return False
    key = (cd, z.device.index, transposed)
    plans = _plans.setdefault(module, {})
    plan = plans.get(key)
    if plan is None or not plan.valid():
        guard = _guard(module)
        if guard is None:
            return False
        plan = host().make_update(guard, module, z, cd, transposed)
        if plan is None:
            return False
        plans[key] = plan
    plan.run(z, out, _masks(z, mask, cd), add, ops.kernel_timer, ops.poison_workspaces)
    return True
