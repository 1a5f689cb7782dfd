"""k_quad (stage-kernel variant 9) where its waves take several groups: its
persistent loop with the loads of one group ahead of the stores of the one
before it, both kinds of register access, a partial last group, and a block
whose last wave has none.

Sizes, in tets, per order: "cached" has more groups than waves run at once (at
most 32,768 tets at N = 1, 24,576 at N = 2, 16,384 above) and registers that
fit the 256 MB cache, "streamed" ones that do not with any epilogue, "idle"
271 groups on 136 blocks of two working waves. All leave two or six elements
in the last group.

Tolerances: as for every FP64 kernel 1e-12 for a few LSERK4 steps and 1e-11 for
KCL frames; compressed LSERK4 steps keep every bit of the one-lane-per-node
kernels; compressed KCL registers 1e-6.
"""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

QUAD = 9
OTHER = {1: 7, 2: 7, 3: 7, 4: 4}
DIMS = {
    "idle": {1: (19, 19, 1), 2: (19, 19, 1), 3: (19, 19, 1), 4: (19, 19, 1)},
    "cached": {1: (23, 23, 23), 2: (19, 17, 17), 3: (15, 15, 15), 4: (15, 15, 13)},
    "streamed": {1: (47, 47, 47), 2: (35, 35, 35), 3: (29, 29, 27), 4: (25, 23, 23)},
}


@pytest.fixture(scope="module")
def ctx():
    from rapidfem_amd import GpuContext

    return GpuContext()


def _setup(order, size):
    import rapidfem_amd as R

    n = DIMS[size][order]
    rng = np.random.default_rng(order)
    mesh = R.structured_box_jittered(*n, 1.0, 1.0, 1.0, 0.1, 3)
    op = R.MaxwellOperator(mesh, order, 0.7, materials={"eps": rng.uniform(1.0, 4.0, (mesh.n_tets, 3))})
    assert op.n_elem % 8 in (2, 6)
    dt = 0.1 / max(n) / (order + 1) ** 2
    print(f"{size}: {op.n_elem} tets, N={order}, {op.n_dof} DOFs", flush=True)
    return op, rng.normal(size=op.n_dof), dt


@pytest.mark.parametrize("size", ["idle", "cached", "streamed"])
@pytest.mark.parametrize("order", [1, 2, 3, 4])
def test_lserk_loop_matches_other_kernels(ctx, order, size):
    import rapidfem_amd as R

    op, y, dt = _setup(order, size)
    b = np.random.default_rng(7).normal(size=op.n_dof)
    runs = {}
    for form, v in (("plain_f64", None), ("fused_f64", QUAD), ("fused_f64c", OTHER[order]), ("fused_f64c", QUAD)):
        g = R.GpuOperator(ctx, op, form)
        if v is not None:
            g.set_variant(v)
            g.poison_lds()
        runs[form, v] = g.transient(ctx, y, dt, 3, 1, R.Drive.vector(b), np.array([0.4, -0.3, 0.2]), record=False,
                                    precision="f64")
        del g
    err = rel_l2(runs["fused_f64", QUAD], runs["plain_f64", None])
    print(f"lserk N={order} {size}: f64 {err:.2e}", flush=True)
    assert err < 1e-12
    assert np.array_equal(runs["fused_f64c", QUAD], runs["fused_f64c", OTHER[order]])


@pytest.mark.parametrize("size", ["idle", "cached", "streamed"])
@pytest.mark.parametrize("order", [1, 2, 3, 4])
def test_kcl_loop_matches_other_kernels(ctx, order, size):
    import rapidfem_amd as R

    op, y, dt = _setup(order, size)
    ctl = R.Controller(atol=1e-3, rtol=1e-3)
    g = R.GpuOperator(ctx, op, "plain_f64")
    want, s = g.transient_kcl(ctx, y, 4 * dt, 1, ctl=ctl, precision="f64")
    del g
    g = R.GpuOperator(ctx, op, "fused_f64c")
    g.set_variant(QUAD)
    for mode in ("f64", "compressed"):
        g.set_kcl_registers(mode)
        g.poison_lds()
        got, st = g.transient_kcl(ctx, y, 4 * dt, 1, ctl=ctl, precision="f64")
        err = rel_l2(got[-1], want[-1])
        print(f"kcl N={order} {size} {mode}: {st.accepted}/{st.rejected}, plain {s.accepted}/{s.rejected}, {err:.2e}",
              flush=True)
        assert (st.accepted, st.rejected) == (s.accepted, s.rejected)
        assert err < (1e-11 if mode == "f64" else 1e-6)
