"""expm and ETD steps at the ends of the Krylov dimension's range (1 to 64),
the normalisation of the start vector, and inputs without a finite norm.

Tolerance: 1e-10 against the oracle's CGS2 as for every FP64 exponential; at a
fixed dimension both span the same Krylov space, and the loss of orthogonality
of the basis (1e-15 after reorthogonalisation) enters once.
"""
import numpy as np
import pytest

from conftest import oracle_desc, rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    from rapidfem_amd import GpuContext

    return GpuContext()


@pytest.fixture(scope="module")
def operators(ctx, oracle):
    from rapidfem_amd import GpuOperator

    xyz, tets = oracle.box_mesh(3, 2, 3, 1.0, 1.0, 1.0, 0.1, 7, True)
    oop = oracle.Operator(xyz, tets, 2, 1.0)
    d, arrs, re_, ex = oracle_desc(oop)
    return oop, GpuOperator.from_desc(ctx, d, "fused_f64", mass=re_["mass"], det=ex["det"])


@pytest.mark.parametrize("m", [1, 2, 63, 64])
@pytest.mark.parametrize("scale", [1.0, 1e-120, 1e120])
def test_dimensions_at_the_ends_match_oracle(ctx, operators, m, scale):
    oop, g = operators
    rng = np.random.default_rng(m)
    y, b = scale * rng.normal(size=oop.n_dof), scale * rng.normal(size=oop.n_dof)
    want, dim = oop.expmv(y, 0.05, m, 0.0)
    assert rel_l2(g.expmv(ctx, y, 0.05, m, 0.0) / scale, want / scale) < 1e-10
    assert g.last_dim == dim == m
    assert rel_l2(g.etd_step(ctx, y, b, 0.05, m, 0.0) / scale, oop.etd_step(y, b, 0.05, m, 0.0) / scale) < 1e-10


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_no_finite_norm_gives_no_finite_result(ctx, operators, bad):
    oop, g = operators
    y = np.random.default_rng(0).normal(size=oop.n_dof)
    y[7] = bad
    assert not np.isfinite(g.expmv(ctx, y, 0.05, 5, 0.0)).any()
    assert g.last_dim == 5
