"""Krylov exponentials where the last columns of the largest bases decide the
result, and start vectors of every scale.

Tolerances: 1e-10 against the oracle's CGS2 as for every FP64 exponential. The
rounding of an apply in FP32 (6e-8) or in three bf16 pieces is amplified by the
products of at most 20 columns; 1e-4 asked between scales, where a vector
outside the FP32 range would leave nothing.
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
def case(oracle):
    xyz, tets = oracle.box_mesh(3, 2, 3, 1.0, 1.0, 1.0, 0.1, 7, True)
    return oracle.Operator(xyz, tets, 2, 1.0)


def _gop(ctx, oop, form):
    from rapidfem_amd import GpuOperator

    d, arrs, re_, ex = oracle_desc(oop)
    return GpuOperator.from_desc(ctx, d, form, mass=re_["mass"], det=ex["det"])


@pytest.mark.parametrize("m", [62, 63, 64])
def test_late_columns_match_oracle(ctx, case, m):
    """At t = 0.8 the oracle's results of m and m - 1 columns differ by about
    2e-5, five orders above the tolerance."""
    rng = np.random.default_rng(63)
    y, b = rng.normal(size=case.n_dof), rng.normal(size=case.n_dof)
    t = 0.8
    want, dim = case.expmv(y, t, m, 0.0)
    less, _ = case.expmv(y, t, m - 1, 0.0)
    want_e, less_e = case.etd_step(y, b, t, m, 0.0), case.etd_step(y, b, t, m - 1, 0.0)
    assert dim == m
    assert rel_l2(less, want) > 1e-6 and rel_l2(less_e, want_e) > 1e-6
    g = _gop(ctx, case, "fused_f64")
    e = rel_l2(g.expmv(ctx, y, t, m, 0.0), want)
    assert g.last_dim == m
    ee = rel_l2(g.etd_step(ctx, y, b, t, m, 0.0), want_e)
    print(f"m={m}: expmv {e:.2e}, etd {ee:.2e}", flush=True)
    assert e < 1e-10 and ee < 1e-10


@pytest.mark.parametrize("scale", [1e-150, 1e-20, 1e20, 1e150])
@pytest.mark.parametrize("form", ["plain_f32", "plain_f64", "fused_f64", "fused_f64c", "fused_bf16x3"])
def test_start_vector_of_any_scale(ctx, case, form, scale):
    y = np.random.default_rng(5).normal(size=case.n_dof)
    g = _gop(ctx, case, form)
    single = form in ("plain_f32", "fused_bf16x3")
    want = g.expmv(ctx, y, 0.05, 20, 0.0) if single else case.expmv(y, 0.05, 20, 0.0)[0]
    e = rel_l2(g.expmv(ctx, scale * y, 0.05, 20, 0.0) / scale, want)
    print(f"{form} scale {scale:g}: {e:.2e}", flush=True)
    assert g.last_dim == 20
    assert e < (1e-4 if single else 1e-10)
