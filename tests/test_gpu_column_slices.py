"""Projections whose workgroups take shares of the output columns (few tiles: csrc/pairproj.hip, in_slices): two and three slices
and the sizes at which one more or one fewer are used, against the general kernels."""
import pytest

from tests import test_gpu_packed_rows as packed


@pytest.mark.gpu
@pytest.mark.parametrize("c_z,mode,n", [(128, "fp32", n) for n in (5, 53, 64, 93, 97, 98, 119, 120)]
                         + [(128, m, n) for m in ("amp", "bf16") for n in (5, 52, 53, 63, 64, 65)]
                         + [(64, m, n) for m in ("amp", "fp32") for n in (52, 64, 65)] + [(256, "amp", n) for n in (52, 53, 64, 65)])
def test_slices(c_z, mode, n, monkeypatch):
    packed.test_updates_equal_the_general_kernels(c_z, mode, n, monkeypatch)
