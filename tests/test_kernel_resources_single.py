"""Scalar registers of the single-solve fused kernels (CPU only, from the built
library's metadata).  Scalars that do not fit are moved through vector lanes in
kernels that are bound by vector issue: the choice of a solve at run time, which
launches shared by several solves need, stays out of the kernel of one solve."""

import pytest

from test_kernel_resources import _kernels, _pick

# k_fused<4, 8, 1, MODE, IQA, X1 = false, PART = 0, DMA = false, MANY = false>:
# spills as built, and room for a compiler's change of mind.
LIMITS = {("0", "0"): 60, ("0", "1"): 115, ("1", "0"): 56, ("1", "1"): 125,
          ("2", "0"): 80, ("2", "1"): 170}


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    return _kernels(tmp_path_factory.mktemp("co"))


@pytest.mark.parametrize("mode,iqa", sorted(LIMITS))
def test_single_solve_kernels_keep_their_scalars(kernels, mode, iqa):
    name = r"7k_fusedILi4ELi8ELi1ELi%sELb%sELb0ELi0ELb0ELb%d"
    single = _pick(kernels, name % (mode, iqa, 0))
    many = _pick(kernels, name % (mode, iqa, 1))
    assert len(single) == 1 and len(many) == 1
    spill = [int(f["sgpr_spill_count"]) for k in (single, many) for f in k.values()]
    assert spill[0] <= LIMITS[mode, iqa] and spill[0] <= spill[1], spill
