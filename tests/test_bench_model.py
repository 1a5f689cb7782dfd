"""What bench.py says about the kernels it times."""
import os
import re

import pytest

from conftest import ROOT

import bench


def test_every_kernel_named_in_the_benchmark_exists():
    src = ""
    csrc = os.path.join(ROOT, "rapidfem_amd", "csrc")
    for f in sorted(os.listdir(csrc)):
        if f.endswith((".hip", ".hpp")):
            with open(os.path.join(csrc, f)) as h:
                src += h.read()
    with open(os.path.join(ROOT, "bench.py")) as h:
        named = set(re.findall(r"\bk_[a-z0-9_]+\b", h.read()))
    assert named
    assert not {k for k in named if not re.search(rf"\b{k}\b\s*\(", src)}


@pytest.mark.parametrize("dim", [1, 2, 40, 64])
def test_krylov_bytes_are_two_basis_sweeps_a_column(dim):
    """Every sweep of an expmv call, column by column, as the kernels' comments
    state it: k_gram2 over cols columns, k_dcgs_update over the j columns before
    q and z (both read and written), one closing product, one combination."""
    n, order = 1000, 3
    read = write = 0
    for j in range(dim):
        cols = j + 2
        read += cols
        read += j + 2
        write += 2
    read += dim + 1
    read += dim
    write += 1
    want = 8.0 * n * (read + write) + dim * n * bench.apply_bytes_per_dof(order)
    assert bench.krylov_bytes(order, n, dim) == want
    # three sweeps a column, as CGS2 with its two middle ones fused takes, move more
    assert dim < 40 or 1.3 * want < 8.0 * n * sum(3 * j + 8 for j in range(dim))
