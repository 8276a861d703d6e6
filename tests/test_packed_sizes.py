"""Elements of a packed weight set: the fragments and, where kernels that keep whole matrices in LDS may be taken (16-bit
arithmetic, 128 channels), the matrices once more; nothing reserved beyond."""
import pytest

from protenix_amd import _lib

F32, BF16, MIXED = _lib.PTX_F32, _lib.PTX_BF16, _lib.PTX_MIXED


@pytest.mark.parametrize("c,hidden,dtype,want", [
    (64, 128, F32, 5 * 64 * 128 + 64 * 64), (64, 128, BF16, 5 * 64 * 128 + 64 * 64), (128, 128, F32, 6 * 128 * 128),
    (128, 128, BF16, 12 * 128 * 128), (128, 128, MIXED, 12 * 128 * 128), (256, 256, BF16, 6 * 256 * 256)])
def test_trimul(c, hidden, dtype, want):
    assert _lib.load().ptx_trimul_packed_elems(c, hidden, dtype) == want


@pytest.mark.parametrize("c,heads,dtype,rows_too", [
    (64, 4, F32, False), (64, 4, BF16, False), (128, 4, F32, False), (128, 4, BF16, True), (128, 4, MIXED, True), (256, 8, BF16, False)])
def test_triattn(c, heads, dtype, rows_too):
    hd = 32 * heads
    want = (4 * hd + 32) * c + c * hd + (5 * c * hd + heads * c if rows_too else 0)     # (the bias' rows fill a tile of 32)
    assert _lib.load().ptx_triattn_packed_elems(c, heads, dtype) == want
