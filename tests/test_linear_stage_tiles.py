"""The workgroups of a linear stage: one per tile of the output, whatever the number of column tiles (they go to the
XCDs in sets of eight), counted on the CPU and, on the GPU, seen to cover every output."""
import ctypes
import math

import pytest
import torch
import torch.nn.functional as F

from protenix_amd import _lib, ops
from tests.util import rel_err, tol

N_OUT = [8, 16, 24, 40, 120, 136, 248, 256, 264, 384, 392, 1536]


@pytest.mark.parametrize("rows", [1, 17, 93, 400, 5000])
@pytest.mark.parametrize("n_out", N_OUT)
def test_one_workgroup_per_tile(rows, n_out):
    lib = _lib.load()
    stage = (ctypes.c_int64 * 32)()
    # (addresses are only looked at for their alignment: nothing is launched)
    rc = lib.ptx_single_linear_stage(ctypes.addressof(stage), 64, 64, None, None, 0, None, 64, None, n_out, 0, rows, 384, n_out, 1, 0)
    assert rc == 0
    kind, n_work, _, tile, row_blocks = (ctypes.c_int32 * 5).from_buffer(stage)
    rm, cn = (16, 16, 32)[tile - 1], (16, 32, 32)[tile - 1]
    assert kind == 1 and row_blocks == -(-rows // rm)
    cols = -(-n_out // cn)
    assert n_work == cols * row_blocks
    # the mapping of linear_stage(): every tile once
    seen = set()
    width = next(w for w in (8, 4, 2, 1) if cols % w == 0)
    for wg in range(n_work):
        group, i = divmod(wg, width * row_blocks)
        seen.add((i // width, width * group + i % width))
    assert seen == {(r, c) for r in range(row_blocks) for c in range(cols)}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows", [5, 93, 1000])
@pytest.mark.parametrize("n_out", N_OUT)
def test_every_output_is_written(rows, n_out, dtype):
    g = torch.Generator().manual_seed(n_out)
    x, w = torch.randn(rows, 64, generator=g).to(dtype), (torch.randn(n_out, 64, generator=g) / math.sqrt(64)).to(dtype)
    nan = torch.full((rows, n_out), float("nan"), device="cuda")
    del nan                                     # (the output is likely made where these were)
    assert rel_err(ops.linear(x.cuda(), w.cuda()), F.linear(x.float(), w.float())) <= tol(dtype)
