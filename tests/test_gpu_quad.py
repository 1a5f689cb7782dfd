"""k_quad (stage-kernel variant 9, eight elements per wave) at the edges of its
groups: element counts around multiples of eight, a wave's first and last
group partial, boundary, port and interior faces mixed, against the oracle.

Tolerances: FP64 sums of at most a few hundred terms of size |A||y| round to
about 1e-14 of the result's norm per apply, 1e-12 asked as for every FP64
kernel; the compressed registers carry 2^-24 of p per stage, 1e-7 asked.
"""
import numpy as np
import pytest

from conftest import oracle_desc, rel_l2

pytestmark = pytest.mark.gpu

QUAD = 9


@pytest.fixture(scope="module")
def ctx():
    from rapidfem_amd import GpuContext

    return GpuContext()


def _submesh_operator(oracle, order, k):
    """The first k tets of a jittered box: any count, walls where tets are
    missing, random materials, losses and ports."""
    xyz, tets = oracle.box_mesh(3, 3, 3, 1.0, 1.0, 1.0, 0.1, 7, True)
    tets = tets.reshape(-1, 4)[:k]
    rng = np.random.default_rng(100 * order + k)
    port = np.where(rng.random(4 * k) < 0.3, 0, -1).astype(np.int32)
    return oracle.Operator(xyz, tets, order, 0.7, eps=rng.uniform(1, 4, (k, 3)), mu=rng.uniform(1, 2, (k, 3)),
                           sigma=rng.uniform(0, 1, k), sigma_m=rng.uniform(0, 1, k), face_port=port)


@pytest.mark.parametrize("order", [1, 2, 3, 4])
@pytest.mark.parametrize("k", [1, 7, 8, 9, 33, 129])
def test_partial_groups_match_oracle(ctx, oracle, order, k):
    from rapidfem_amd import Drive, GpuOperator

    oop = _submesh_operator(oracle, order, k)
    n = oop.n_dof
    rng = np.random.default_rng(k)
    y, b = rng.normal(size=n), rng.normal(size=n)
    wave = np.array([0.4, -0.3, 0.2])
    dt = 0.002
    want = oop.apply(y)
    want_vec = oop.lserk(y, dt, 3, ("vector", b), wave)
    want_pt = oop.lserk(y, dt, 3, ("point", n - 1), wave)
    d, arrs, re_, ex = oracle_desc(oop)
    for form in ("fused_f64", "fused_f64c"):
        g = GpuOperator.from_desc(ctx, d, form, mass=re_["mass"], det=ex["det"])
        g.set_variant(QUAD)
        g.poison_lds()
        e = [rel_l2(g.apply_f64(y), want)]
        for drive, w in ((Drive.vector(b), want_vec), (Drive.point(n - 1), want_pt)):
            g.poison_lds()
            e.append(rel_l2(g.transient(ctx, y, dt, 3, 1, drive, wave, record=False, precision="f64"), w))
        print(f"quad order={order} K={k} {form}: apply {e[0]:.2e}, vector {e[1]:.2e}, point {e[2]:.2e}", flush=True)
        assert e[0] < 1e-12
        assert max(e[1:]) < (1e-7 if form == "fused_f64c" else 1e-12)


@pytest.mark.parametrize("order", [1, 2, 3, 4])
@pytest.mark.parametrize("k", [1, 9, 129])
def test_kcl_on_partial_groups_matches_oracle(ctx, oracle, order, k):
    """The fused KCL update (FP64 and compressed registers), whose error norm
    sums one partial per wave, idle waves included: FP64 takes the oracle's
    accept/reject sequence; either meets the controller's states."""
    from rapidfem_amd import Controller, GpuOperator

    oop = _submesh_operator(oracle, order, k)
    y0 = np.random.default_rng(k).normal(size=oop.n_dof)
    ctl, octl = Controller(atol=1e-7, rtol=1e-5), oracle.Controller.default()
    octl.atol, octl.rtol = 1e-7, 1e-5
    want, acc, rej, _, _ = oop.adaptive(y0, 0.01, 2, octl)
    d, arrs, re_, ex = oracle_desc(oop)
    g = GpuOperator.from_desc(ctx, d, "fused_f64c", mass=re_["mass"], det=ex["det"])
    g.set_variant(QUAD)
    for mode in ("f64", "compressed"):
        g.set_kcl_registers(mode)
        g.poison_lds()
        traj, st = g.transient_kcl(ctx, y0, 0.01, 2, ctl=ctl, precision="f64")
        err = rel_l2(traj[-1], want)
        print(f"quad kcl order={order} K={k} {mode}: {st.accepted}/{st.rejected}, oracle {acc}/{rej}, {err:.2e}",
              flush=True)
        if mode == "f64":
            assert (st.accepted, st.rejected) == (acc, rej)
        assert err < (1e-11 if mode == "f64" else 1e-6)


@pytest.mark.parametrize("alpha", [1.0, 0.7, 0.0])
@pytest.mark.parametrize("order, other", [(1, 7), (2, 7), (3, 7), (4, 4)])
def test_compressed_registers_keep_every_bit(ctx, oracle, order, other, alpha):
    """With compressed registers k_quad takes every sum in the order of the
    one-lane-per-node kernels: 40 steps leave the same bits. In the second run
    a held source -A y leaves the rounding of the first stage's right-hand side
    as the whole of p, so its last FP64 bit shows."""
    from rapidfem_amd import Drive, GpuOperator

    k = 129
    xyz, tets = oracle.box_mesh(3, 3, 3, 1.0, 1.0, 1.0, 0.1, 7, True)
    rng = np.random.default_rng(order)
    port = np.where(rng.random(4 * k) < 0.3, 0, -1).astype(np.int32)
    oop = oracle.Operator(xyz, tets.reshape(-1, 4)[:k], order, alpha, eps=rng.uniform(1, 4, (k, 3)),
                          sigma=rng.uniform(0, 1, k), face_port=port)
    y = rng.normal(size=oop.n_dof)
    d, arrs, re_, ex = oracle_desc(oop)
    g = GpuOperator.from_desc(ctx, d, "fused_f64c", mass=re_["mass"], det=ex["det"])
    got = []
    for v in (other, QUAD):
        g.set_variant(v)
        g.poison_lds()
        got.append(g.transient(ctx, y, 0.001, 40, 1, Drive.point(3), np.linspace(0, 1, 40), record=False,
                               precision="f64"))
    assert np.array_equal(got[0], got[1])
    y = np.ldexp(y.astype(np.float32).astype(np.float64), -60)
    src = -g.apply_f64(y)
    got = []
    for v in (other, QUAD):
        g.set_variant(v)
        got.append(g.transient(ctx, y, 1e8, 1, 1, Drive.vector(src), np.ones(1), record=False, precision="f64"))
    assert np.isfinite(got[0]).all() and np.array_equal(got[0], got[1])
