"""The work a user of rapidfem_amd has it do, as cases that can be timed and
checked: one operator apply, explicit LSERK4 transients at every order, the
adaptive KCL stepper, the Krylov exponentials, port-driven meshes advanced
together and the sparse export, on jittered Kuhn boxes with the materials,
walls and drives of the package's workloads.

A case is a dict of plain values:
  kind      apply | lserk | probes | kcl | expmv | etd | adaptive | batch | sparse
  nx,ny,nz  cells of the unit-width box (six tets each)
  order     polynomial order 1..4
  form      fused_f64 (the default form) or fused_f64c (compressed registers)
  medium    vacuum | block (dielectric, eps 2 to 6) | slab (thin lossy slab, graded cells) | debye (dispersive block)
  drive     free | point (one DOF) | port (TE10 port pattern; batch only)
  steps     LSERK4 steps, KCL frames or exponential steps, as the kind has it

`exact` computes the same outputs in 64 bits with plain torch: its own
reference element (rational arithmetic), face matching, flux and steppers,
for the exponentials a Taylor series over short substeps.
"""
from __future__ import annotations

import math
from fractions import Fraction
from functools import lru_cache

import numpy as np
import torch

import rapidfem_amd as R
from rapidfem_amd.maxwell import boundary_faces_on_plane, port_face_data
from rapidfem_amd.proposer import WEIGHTS, ExpController, Proposer

TOL_KRYLOV = 1e-10  # the session's a-posteriori tolerance of expmv / etd_step
N_PROBES = 64


def _case(name, kind, nx, ny, nz, order, form="fused_f64", medium="vacuum", drive="free", steps=1, **more):
    return dict(name=name, kind=kind, nx=nx, ny=ny, nz=nz, order=order, form=form, medium=medium, drive=drive,
                steps=steps, **more)


def listed():
    return [
        # One operator apply between host vectors on the smallest mesh in use (1,296 tets, N=2):
        # what an outer Krylov or eigenvalue loop of the caller's own pays per call.
        _case("apply_small_n2", "apply", 6, 6, 6, 2),
        # The cavity transient (1,296 tets, N=2), a point source, 64 probe DOFs recorded every step:
        # thousands of very short launches.
        _case("probes_small_n2", "probes", 6, 6, 6, 2, drive="point", steps=300),
        # A first-order run on a mesh of a user's own, odd sizes (27,030 tets).
        _case("lserk_n1", "lserk", 17, 5, 53, 1, steps=200),
        # The benchmark stepper: 324,000 tets, N=3, dielectric block, compressed registers.
        _case("lserk_block_n3_f64c", "lserk", 60, 30, 30, 3, "fused_f64c", "block", steps=100),
        # The default form at N=3 on the graded lossy-slab mesh, ragged sizes (85,176 tets).
        _case("lserk_slab_n3_f64", "lserk", 26, 26, 21, 3, "fused_f64", "slab", "point", steps=100),
        # Fourth order with compressed registers, cavity modes (470,400 tets, 98.8M DOFs).
        _case("lserk_modes_n4_f64c", "lserk", 40, 40, 49, 4, "fused_f64c", steps=30),
        # A dispersive (Debye) block at second order, compressed registers (72,912 tets).
        _case("lserk_debye_n2_f64c", "lserk", 31, 28, 14, 2, "fused_f64c", "debye", steps=150),
        # The adaptive KCL stepper with its default FP64 registers, N=3, dielectric block (100,800 tets).
        _case("kcl_block_n3", "kcl", 30, 28, 20, 3, medium="block", steps=3, cfl=4.0),
        # exp(tA) v at the session's dimension and tolerance on the stiff slab mesh (201,600 tets, N=3).
        _case("expmv_slab_n3", "expmv", 40, 30, 28, 3, medium="slab", steps=1, m=40, cfl=5.0),
        # The learned (h, m) exponential on a slab mesh a quarter that size.
        _case("adaptive_slab_n3", "adaptive", 24, 22, 17, 3, medium="slab", steps=1, cfl=50.0),
        # Port excitations of uneven meshes at orders 2, 3 and 4 advanced together in one graph.
        _case("batch_ports", "batch", 19, 17, 20, 2, "fused_f64c", "block", "port", steps=60, meshes=3),
        # The state-space matrix of a small second-order model, downloaded.
        _case("sparse_n2", "sparse", 9, 8, 7, 2, medium="block"),
    ]


def _dims(rng, lo, hi):
    """Cells of a box with between lo and hi tets, log-uniform, uneven sides."""
    c = (math.exp(rng.uniform(math.log(lo), math.log(hi))) / 6.0) ** (1.0 / 3.0)
    a = rng.uniform(0.7, 1.4)
    b = rng.uniform(0.7, 1.0)
    nx, ny = max(2, round(c * a)), max(2, round(c * b))
    return nx, ny, max(2, min(round(c ** 3 / (nx * ny)), int(hi / (6 * nx * ny))))


def draw(rng):
    kind = rng.choice(["apply", "probes", "lserk", "lserk", "lserk", "lserk", "kcl", "expmv", "etd", "adaptive",
                       "batch", "sparse"])
    order = rng.choice([1, 2, 3, 4])
    form = rng.choice(["fused_f64", "fused_f64c"])
    medium = rng.choice(["vacuum", "block", "slab", "debye"])
    drive = rng.choice(["free", "point"])
    most = {1: 400_000, 2: 300_000, 3: 200_000, 4: 150_000}[order]
    c = dict(kind=kind, order=order, form=form, medium=medium, drive=drive, steps=1)
    if kind == "apply":
        c.update(drive="free", form="fused_f64")
    elif kind == "probes":
        c["steps"] = rng.randrange(50, 200)
        most //= 4
    elif kind == "lserk":
        c["steps"] = rng.randrange(40, 120)
    elif kind == "kcl":
        c.update(steps=2, cfl=rng.uniform(1.5, 4.0), form="fused_f64")
        most //= 2
    elif kind in ("expmv", "etd"):
        c.update(form="fused_f64", m=rng.choice([16, 24, 30, 40]), cfl=rng.uniform(1.0, 5.0),
                 drive="free" if kind == "expmv" else "point")
        most //= 2
    elif kind == "adaptive":
        c.update(form="fused_f64", cfl=rng.uniform(15.0, 60.0), drive="free", medium=rng.choice(["slab", "block"]))
        most //= 6
    elif kind == "batch":
        c.update(order=2, drive="port", medium="block", steps=2 * rng.randrange(10, 30), meshes=rng.choice([2, 3, 4]))
        most = 40_000
    else:
        c.update(form="fused_f64", drive="free", medium="block")
        most = {1: 8000, 2: 3000, 3: 1000, 4: 500}[order]
    c["nx"], c["ny"], c["nz"] = _dims(rng, most / 100 if kind != "sparse" else 60, most)
    return c


# ---- the mesh, medium and fields of a case --------------------------------------------------


def _mesh(case, seed):
    """Nodes (n, 3) and ascending tets (K, 4) of the case's box: cells of unit width scaled to x in
    [0, nx/ny], interior nodes moved by up to 10 % of a cell; a slab medium grades the cells along x."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    # one mesh per sparse case: which entries it stores follows from the round-off on its mesh
    rng = np.random.default_rng([seed if case["kind"] != "sparse" else 0, 1])
    g = np.stack(np.meshgrid(np.arange(nz + 1.0), np.arange(ny + 1.0), np.arange(nx + 1.0), indexing="ij"), -1)
    g = g.reshape(-1, 3)[:, ::-1].copy()
    n = np.array([nx, ny, nz], np.float64)
    inside = (g > 0) & (g < n)
    if case["medium"] != "slab":
        g += np.where(inside, rng.uniform(-0.1, 0.1, g.shape), 0.0)
    g /= n[1]
    if case["medium"] == "slab":
        x = (np.arange(nx) + 0.5) / nx
        w = 1.0 / (1.0 + 19.0 * np.exp(-(((x - 0.45) / 0.06) ** 2)))
        xs = np.concatenate([[0.0], np.cumsum(w)]) * (nx / ny) / w.sum()
        g[:, 0] = xs[np.rint(g[:, 0] * ny).astype(np.int64)]
    kuhn = np.array([[0, 1, 3, 7], [0, 3, 2, 7], [0, 2, 6, 7], [0, 6, 4, 7], [0, 4, 5, 7], [0, 5, 1, 7]])
    corner = (kuhn & 1) + ((kuhn >> 1) & 1) * (nx + 1) + ((kuhn >> 2) & 1) * (nx + 1) * (ny + 1)
    k, j, i = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    c0 = ((k * (ny + 1) + j) * (nx + 1) + i).reshape(-1, 1, 1)
    return g, np.sort((c0 + corner).reshape(-1, 4), axis=1).astype(np.int64)


def _medium(case, nodes, tets, seed):
    """eps (K,), sigma (K,) and the Debye elements of the case's medium."""
    x = ((np.arange(len(tets)) // 6) % case["nx"] + 0.5) / case["nx"]  # by cell, whatever the jitter
    if case["medium"] == "slab":
        x = nodes[tets].mean(axis=1)[:, 0] * case["ny"] / case["nx"]
    eps, sigma, debye = np.ones(len(tets)), np.zeros(len(tets)), np.zeros(0, np.int64)
    if case["medium"] == "block":
        eps[(x >= 0.4) & (x <= 0.6)] = np.random.default_rng([seed, 6]).uniform(2.0, 6.0)
    elif case["medium"] == "slab":
        slab = np.abs(x - 0.45) <= 0.03
        eps[slab], sigma[slab] = 10.0, 50.0
    elif case["medium"] == "debye":
        debye = np.nonzero((x >= 0.45) & (x <= 0.55))[0]
        eps[debye] = 2.0
    return eps, sigma, debye


DEBYE = dict(eps_inf=2.0, eps_static=6.0, tau=0.2)


def _dt(nodes, tets, order):
    """A stable LSERK4 step: the smallest element height over the order."""
    g, _ = _gradients(nodes, tets)
    return 0.35 / (np.sqrt((g ** 2).sum(-1)).max() * (order + 1) ** 2)


def _gradients(nodes, tets):
    """Outward face vectors g_f = -grad(lambda_opposite) (K, 4, 3) and J^-1 (K, 3, 3)."""
    v = nodes[tets]
    jinv = np.linalg.inv(np.swapaxes(v[:, 1:] - v[:, :1], 1, 2))
    return np.stack([-jinv[:, 2], -jinv[:, 0], -jinv[:, 1], jinv.sum(1)], axis=1), jinv


def _field(case, x, lengths, seed):
    """A start field at the points x (n, 3): Gaussian pulse plus three cavity modes, seeded."""
    rng = np.random.default_rng([seed, 2])
    out = np.zeros((len(x), 6))
    c = rng.uniform(0.2, 0.8, 3) * lengths
    r2 = ((x - c) ** 2).sum(1)
    out[:, 0] = np.exp(-r2 / 0.02) * np.sin(10.0 * math.pi * x[:, 0])
    for axis, a in zip(rng.permutation(3), rng.normal(size=3)):
        u, v = (axis + 1) % 3, (axis + 2) % 3
        out[:, axis] += a * np.sin(math.pi * x[:, u] / lengths[u]) * np.sin(math.pi * x[:, v] / lengths[v])
        out[:, 3 + axis] += 0.3 * a * np.cos(math.pi * x[:, u] / lengths[u]) * np.cos(math.pi * x[:, v] / lengths[v])
    return out


def _start(case, nodes, tets, order, seed, n_debye):
    """The start state in the framework's layout, (K, Np, 6) flattened plus a zero P block."""
    lengths = nodes.max(axis=0)
    ijk = np.array(_element(order)["ijk"], np.float64) / order
    bary = np.concatenate([1.0 - ijk.sum(1, keepdims=True), ijk], axis=1)
    y = np.zeros(len(tets) * len(ijk) * 6 + 3 * len(ijk) * n_debye)
    step = 1 << 16
    for a in range(0, len(tets), step):
        x = (bary @ nodes[tets[a:a + step]]).reshape(-1, 3)
        f = _field(case, x, lengths, seed)
        y[a * len(ijk) * 6:a * len(ijk) * 6 + f.size] = f.reshape(-1)
    return y


def _wave(case, seed, n, dt):
    """A modulated Gaussian pulse sampled at n steps of dt."""
    f0 = np.random.default_rng([seed, 3]).uniform(3.0, 8.0)
    t = np.arange(n) * dt - 0.25 * n * dt
    return np.exp(-((t / (0.3 * n * dt)) ** 2)) * np.cos(2.0 * math.pi * f0 * t)


def _source_dof(case, n_eh, seed):
    return int(np.random.default_rng([seed, 4]).integers(n_eh))


def _horizon(case, dt):
    return case["cfl"] * dt * 8.0


def _sub_cases(case):
    """The meshes of a batch: orders 2, 3, 4 in turn, uneven sizes."""
    return [dict(case, order=2 + b % 3, nx=max(2, case["nx"] - 3 * b), nz=max(2, case["nz"] - 2 * b))
            for b in range(case["meshes"])]


def _port_profile(lengths):
    """TE10-shaped incident wave on the wall x = 0: (e_t, h_t) at points (n, 3)."""

    def profile(x):
        e, h = np.zeros_like(x), np.zeros_like(x)
        e[:, 2] = np.sin(math.pi * x[:, 1] / lengths[1])
        h[:, 1] = -e[:, 2]
        return e, h

    return profile


def _operator(case, seed, ports=False):
    nodes, tets = _mesh(case, seed)
    eps, sigma, debye = _medium(case, nodes, tets, seed)
    mats = None if case["medium"] == "vacuum" else {"eps": np.repeat(eps[:, None], 3, axis=1), "sigma": sigma}
    disp = [(int(e), R.DebyeMaterial(**DEBYE)) for e in debye]
    face_port = None
    if ports:
        face_port = np.full((len(tets), 4), -1, np.int32)
        on = np.abs(nodes[tets][..., 0]) < 1e-9
        e = np.nonzero(on.sum(1) == 3)[0]
        # local faces 0..3 lie opposite the vertices 3, 1, 2, 0
        face_port[e, np.array([3, 1, 2, 0])[np.argmin(on[e], axis=1)]] = 0
    op = R.MaxwellOperator(R.Mesh(nodes, tets), case["order"], 1.0, materials=mats, face_port=face_port,
                           dispersive=disp)
    return op, nodes, tets, len(debye)


def prepare(case, seed):
    if case["kind"] == "batch":
        ctx = R.GpuContext()
        subs = [_prepare_batch(ctx, c, seed + 1000 * b) for b, c in enumerate(_sub_cases(case))]
        return dict(case=case, subs=subs, ops=[s["g"] for s in subs], dts=[s["dt"] for s in subs],
                    waves=[s["wave"] for s in subs])
    op, nodes, tets, nd = _operator(case, seed)
    ctx = R.GpuContext()
    s = dict(case=case, op=op, ctx=ctx, dt=_dt(nodes, tets, case["order"]))
    if case["kind"] == "sparse":
        return s
    s["y"] = _start(case, nodes, tets, case["order"], seed, nd)
    s["g"] = R.GpuOperator(ctx, op, case["form"])
    n_eh = len(s["y"]) - 3 * op.re.n_nodes * nd
    s["drive"], s["wave"] = None, None
    if case["drive"] == "point":
        s["drive"] = R.Drive.point(_source_dof(case, n_eh, seed))
        s["wave"] = _wave(case, seed, case["steps"], s["dt"])
    if case["kind"] == "probes":
        s["probes"] = np.random.default_rng([seed, 5]).integers(0, n_eh, N_PROBES)
    if case["kind"] == "etd":
        s["b"] = np.zeros(len(s["y"]))
        s["b"][s["drive"].dof] = 1.0
    if case["kind"] == "adaptive":
        s["ctl"] = ExpController(tol=1e-6, h_scale=s["dt"])
        s["proposer"] = Proposer(ctx)
        s["proposer"].load(WEIGHTS)
    return s


def _prepare_batch(ctx, case, seed):
    op, nodes, tets, _ = _operator(case, seed, ports=True)
    g = R.GpuOperator(ctx, op, case["form"])
    faces = boundary_faces_on_plane(op, 0, 0.0)
    g.set_port(0, *port_face_data(op, faces, _port_profile(nodes.max(axis=0))))
    g.port_source(0, download=False)
    dt = _dt(nodes, tets, case["order"])
    return dict(g=g, dt=dt, y=_start(case, nodes, tets, case["order"], seed, 0),
                wave=_wave(case, seed, case["steps"], dt))


def run(s):
    case = s["case"]
    kind, steps = case["kind"], case["steps"]
    if kind == "apply":
        return s["g"].apply_f64(s["y"])
    if kind == "lserk":
        return s["g"].transient(s["ctx"], s["y"], s["dt"], steps, 1, s["drive"], s["wave"], record=False,
                                precision="f64")
    if kind == "probes":
        return s["g"].transient_probes(s["ctx"], s["y"], s["dt"], steps, s["probes"], 1, s["drive"], s["wave"])
    if kind == "kcl":
        return s["g"].transient_kcl(s["ctx"], s["y"], _horizon(case, s["dt"]), steps, s["drive"], s["wave"],
                                    precision="f64")[0]
    if kind == "expmv":
        return s["g"].expmv(s["ctx"], s["y"], _horizon(case, s["dt"]), case["m"], TOL_KRYLOV)
    if kind == "etd":
        return s["g"].etd_step(s["ctx"], s["y"], s["b"], _horizon(case, s["dt"]), case["m"], TOL_KRYLOV)
    if kind == "adaptive":
        return s["g"].expmv_adaptive(s["ctx"], s["y"], 8.0 * case["cfl"] * s["dt"], s["ctl"], s["proposer"])[0]
    if kind == "batch":
        for sub in s["subs"]:
            sub["g"].state_load(sub["y"])
        R.batch_lserk_ports(s["ops"], s["dts"], steps, s["waves"])
        return [sub["g"].state_store() for sub in s["subs"]]
    m = R.assemble_sparse(s["ctx"], s["op"])
    return m.row_ptr, m.col_idx, m.values


# ---- what a pass cannot do without ------------------------------------------------------------


def _apply_work(case, state_bytes):
    """Bytes and flops of one fused apply or stage: the state, J^-1, face codes and material index per
    element; the volume products, the flux, LIFT, the materials and the update."""
    p = case["order"]
    np_, nfp = (p + 1) * (p + 2) * (p + 3) // 6, (p + 1) * (p + 2) // 2
    k = 6 * case["nx"] * case["ny"] * case["nz"]
    flops = 36 * np_ ** 2 + 114 * np_ + 78 * 4 * nfp + 48 * np_ * nfp + 18 * np_ + 30 * np_
    return k * (state_bytes * 6 * np_ + 92.0), float(k * flops), 6 * np_ * k


def work(case):
    kind, steps = case["kind"], case["steps"]
    if kind == "batch":
        parts = [work(dict(c, kind="lserk")) for c in _sub_cases(case)]
        return {q: sum(w[q] for w in parts) for q in ("bytes", "flops")}
    # y read and written, p read and written: FP64, or f32 + bf16 and f32
    state = 20.0 if case["form"] == "fused_f64c" else 32.0
    b, f, n = _apply_work(case, state)
    ba, fa, _ = _apply_work(case, 16.0)
    if kind == "apply":
        return {"bytes": ba, "flops": fa}
    if kind in ("lserk", "probes"):
        return {"bytes": 16.0 * n + 5 * steps * b, "flops": 5 * steps * f}
    if kind == "kcl":
        # y, err and the stage input read and written in every stage of about 2.5 cfl substeps a frame
        sub = 5 * steps * max(1.0, 2.5 * case["cfl"])
        return {"bytes": 16.0 * n + sub * (ba + 32.0 * n), "flops": sub * (fa + 10.0 * n)}
    if kind in ("expmv", "etd"):
        # about 8 + 4.5 cfl columns reach the tolerance, each projected on the earlier ones and
        # updated by them: one read of the basis for either
        m = min(case["m"], 8.0 + 4.5 * case["cfl"])
        return {"bytes": m * ba + 8.0 * n * (m * m + 2 * m), "flops": m * fa + 4.0 * n * m * m}
    if kind == "adaptive":
        # bases of about 20 columns, each taking the state about 5 CFL steps on
        r, m = max(1.0, case["cfl"] / 5.0), 20
        return {"bytes": r * (m * ba + 8.0 * n * (m * m + 2 * m)), "flops": r * (m * fa + 4.0 * n * m * m)}
    p = case["order"]
    np_, nfp = (p + 1) * (p + 2) * (p + 3) // 6, (p + 1) * (p + 2) // 2
    nnz = 0.6 * n * (4.0 * np_ + 20.0 * nfp)
    return {"bytes": 16.0 * nnz + 8.0 * n, "flops": 30.0 * nnz}


# ---- the same outputs in 64 bits, in plain torch ----------------------------------------------


def _solve(a, b):
    """a^-1 b over the rationals (lists of rows of Fractions)."""
    n = len(a)
    m = [list(r) + list(q) for r, q in zip(a, b)]
    for c in range(n):
        piv = next(r for r in range(c, n) if m[r][c] != 0)
        m[c], m[piv] = m[piv], m[c]
        d = m[c][c]
        m[c] = [v / d for v in m[c]]
        for r in range(n):
            if r != c and m[r][c] != 0:
                f = m[r][c]
                m[r] = [v - f * w for v, w in zip(m[r], m[c])]
    return [r[n:] for r in m]


def _mul(a, b):
    cols = list(zip(*b))
    return [[sum((x * y for x, y in zip(r, c) if x and y), Fraction(0)) for c in cols] for r in a]


@lru_cache(maxsize=None)
def _element(p):
    """Equispaced nodal element of order p: node multi-indices, D_r, D_s, D_t, and LIFT whose columns are
    the face nodes in `faces` order (each face's nodes sorted by their barycentric indices)."""
    ijk = [(i, j, k) for i in range(p + 1) for j in range(p + 1 - i) for k in range(p + 1 - i - j)]
    mono = [(a, b, d - a - b) for d in range(p + 1) for a in range(d + 1) for b in range(d + 1 - a)]
    n = len(ijk)
    eye = [[Fraction(int(i == j)) for j in range(n)] for i in range(n)]
    x = [[Fraction(v, p) for v in q] for q in ijk]

    def ev(m, q):
        return q[0] ** m[0] * q[1] ** m[1] * q[2] ** m[2]

    def dev(m, q, a):
        return m[a] * ev([e - (t == a) for t, e in enumerate(m)], q) if m[a] else Fraction(0)

    coef = _solve([[ev(m, q) for m in mono] for q in x], eye)
    d = [np.array(_mul([[dev(m, q, a) for m in mono] for q in x], coef), np.float64) for a in range(3)]
    fac = math.factorial
    gram = [[Fraction(fac(a[0] + b[0]) * fac(a[1] + b[1]) * fac(a[2] + b[2]), fac(sum(a) + sum(b) + 3))
             for b in mono] for a in mono]
    mass = _mul(_mul([list(r) for r in zip(*coef)], gram), coef)
    # faces by the barycentric index that vanishes on them: vertices 3, 1, 2, 0
    bary = [(p - sum(q),) + q for q in ijk]
    faces, emat = [], [[Fraction(0)] * (4 * (p + 1) * (p + 2) // 2) for _ in range(n)]
    m2 = [(a, t - a) for t in range(p + 1) for a in range(t + 1)]
    for f, opp in enumerate((3, 1, 2, 0)):
        rest = [v for v in range(4) if v != opp]
        fn = sorted((q for q in range(n) if bary[q][opp] == 0), key=lambda q: [bary[q][v] for v in rest])
        uv = [[Fraction(bary[q][v], p) for v in rest[1:]] for q in fn]
        c2 = _solve([[u[0] ** a * u[1] ** b for a, b in m2] for u in uv],
                    [[Fraction(int(i == j)) for j in range(len(fn))] for i in range(len(fn))])
        g2 = [[Fraction(fac(a + c) * fac(b + e), fac(a + b + c + e + 2)) for c, e in m2] for a, b in m2]
        mf = _mul(_mul([list(r) for r in zip(*c2)], g2), c2)
        for i, q in enumerate(fn):
            for j in range(len(fn)):
                emat[q][f * len(fn) + j] = mf[i][j]
        faces.append(fn)
    return dict(ijk=ijk, D=d, lift=np.array(_solve(mass, emat), np.float64), faces=faces)


class _Exact:
    """The DG Maxwell operator in float64 torch on vectors u (Np, 6, K); Debye P blocks (Np, 3, n_debye)."""

    def __init__(self, case, seed, ports=False):
        self.case, self.p = case, case["order"]
        nodes, tets = _mesh(case, seed)
        self.nodes, self.tets = nodes, tets
        eps, sigma, debye = _medium(case, nodes, tets, seed)
        el = _element(self.p)
        dev = "cuda" if torch.cuda.is_available() else "cpu"

        def t(a, kind=torch.float64):
            return torch.as_tensor(np.ascontiguousarray(a), dtype=kind, device=dev)

        self.K, self.np_ = len(tets), len(el["ijk"])
        self.nfp = len(el["faces"][0])
        self.D = t(np.concatenate(el["D"]))
        self.lift, self.faces = t(el["lift"]), t(np.array(el["faces"]), torch.int64)
        g, jinv = _gradients(nodes, tets)
        size = np.sqrt((g ** 2).sum(-1))
        self.n, self.cf = t((g / size[..., None]).transpose(1, 2, 0)), t(0.5 * size.T)  # (4, 3, K), (4, K)
        self.jinv = t(jinv.transpose(1, 2, 0))  # (3 ref, 3 phys, K)
        self.inv_eps, self.sig = t(1.0 / eps), t(sigma / eps)
        self.debye = t(debye, torch.int64)
        self._pair(t(tets, torch.int64))
        self.port = None
        if ports:
            wall = np.stack([(np.abs(nodes[tets][:, [v for v in range(4) if v != o], 0]) < 1e-9).all(1)
                             for o in (3, 1, 2, 0)])
            self.port = t(wall, torch.bool)  # (4, K)
            ijk = np.array(el["ijk"], np.float64) / self.p
            bary = t(np.concatenate([1.0 - ijk.sum(1, keepdims=True), ijk], axis=1))
            x = torch.einsum("nv,kvd->ndk", bary, t(nodes[tets]))
            self.inc = torch.zeros(self.np_, 6, self.K, dtype=torch.float64, device=dev)
            self.inc[:, 2] = torch.sin(math.pi * x[:, 1] / nodes[:, 1].max())
            self.inc[:, 4] = -self.inc[:, 2]

    def _pair(self, tets):
        """Neighbour element and its local face behind every face (element itself on a wall)."""
        tri = torch.stack([tets[:, [v for v in range(4) if v != o]] for o in (3, 1, 2, 0)])  # (4, K, 3), ascending
        n = int(tets.max()) + 1
        key = ((tri[..., 0] * n + tri[..., 1]) * n + tri[..., 2]).reshape(-1)
        key, order = torch.sort(key)
        same = torch.nonzero(key[1:] == key[:-1]).reshape(-1)
        a, b = order[same], order[same + 1]
        other = torch.full_like(order, -1)
        other[a], other[b] = b, a
        other = other.reshape(4, self.K)
        self.wall = other < 0
        own = torch.arange(self.K, device=tets.device)
        self.nbr = torch.where(self.wall, own, other % self.K)
        self.nlf = torch.where(self.wall, 0, other // self.K)

    def vec(self, y):
        """Framework layout -> (u, P)."""
        y = torch.as_tensor(y, dtype=torch.float64, device=self.D.device)
        n = self.K * self.np_ * 6
        return [y[:n].reshape(self.K, self.np_, 6).permute(1, 2, 0).contiguous(),
                y[n:].reshape(-1, self.np_, 3).permute(1, 2, 0).contiguous()]

    def flat(self, v):
        return torch.cat([v[0].permute(2, 0, 1).reshape(-1), v[1].permute(2, 0, 1).reshape(-1)]).cpu().numpy()

    def apply(self, v, inc=0.0):
        """A v, with the port's incident wave at amplitude inc (or a point drive added by the caller)."""
        u, pol = v
        r = (self.D @ u.reshape(self.np_, -1)).reshape(3, self.np_, 6, self.K)
        acc = torch.empty_like(u)
        for c in range(3):
            a, b = (c + 1) % 3, (c + 2) % 3
            for f, s in ((3, 1.0), (0, -1.0)):  # dE = curl H, dH = -curl E
                dab = sum(self.jinv[k, a] * r[k, :, f + b] - self.jinv[k, b] * r[k, :, f + a] for k in range(3))
                acc[:, 3 - f + c] = s * dab
        del r
        flux = torch.empty(4 * self.nfp, 6, self.K, dtype=u.dtype, device=u.device)
        comp = torch.arange(6, device=u.device)[None, :, None]
        for f in range(4):
            n = self.n[f]
            own = u[self.faces[f]]
            jump = own - u[self.faces[self.nlf[f]].T[:, None, :], comp, self.nbr[f][None, None, :]]
            e, h = own[:, :3], own[:, 3:]
            en, hn = (e * n).sum(1, keepdim=True) * n, (h * n).sum(1, keepdim=True) * n
            jump = torch.where(self.wall[f], torch.cat([2.0 * (e - en), 2.0 * hn], dim=1), jump)
            if self.port is not None:
                jump = torch.where(self.port[f], own - inc * self.inc[self.faces[f]], jump)
            je, jh = jump[:, :3], jump[:, 3:]

            def cross(w):
                return torch.stack([n[1] * w[:, 2] - n[2] * w[:, 1], n[2] * w[:, 0] - n[0] * w[:, 2],
                                    n[0] * w[:, 1] - n[1] * w[:, 0]], dim=1)

            ce, ch = cross(je), cross(jh)
            flux[f * self.nfp:(f + 1) * self.nfp] = self.cf[f] * torch.cat([cross(ce) - ch, cross(ch) + ce], dim=1)
        acc += (self.lift @ flux.reshape(4 * self.nfp, -1)).reshape(self.np_, 6, self.K)
        acc[:, :3] = acc[:, :3] * self.inv_eps - self.sig * u[:, :3]
        dp = pol
        if len(self.debye):
            delta = DEBYE["eps_static"] - DEBYE["eps_inf"]
            dp = (delta * u[:, :3, self.debye] - pol) / DEBYE["tau"]
            acc[:, :3, self.debye] -= dp / DEBYE["eps_inf"]
        return [acc, dp]

    def add_point(self, v, dof, g):
        e, r = divmod(dof, self.np_ * 6)
        v[0][r // 6, r % 6, e] += g

    def lserk(self, v, dt, steps, force, each=None):
        a = (0.0, -567301805773 / 1357537059087, -2404267990393 / 2016746695238, -3550918686646 / 2091501179385,
             -1275806237668 / 842570457699)
        b = (1432997174477 / 9575080441755, 5161836677717 / 13612068292357, 1720146321549 / 2090206949498,
             3134564353537 / 4481467310338, 2277821191437 / 14882151754819)
        w = [torch.zeros_like(x) for x in v]
        for s in range(steps):
            for q in range(5):
                k = force(v, s)
                for x, y, z in zip(w, v, k):
                    x.mul_(a[q]).add_(z, alpha=dt)
                    y.add_(x, alpha=b[q])
            if each:
                each(s, v)
        return v

    def flow(self, v, t, force):
        """y' = A y + b over [0, t]: a Taylor series of A over substeps of |h A| about 1. force(v) is
        A v + b and force(v, False) is A v."""
        x = [torch.randn_like(q) for q in v]
        for _ in range(6):
            size = math.sqrt(sum(float((q * q).sum()) for q in x))
            x = self.apply([q / size for q in x])
        rho = math.sqrt(sum(float((q * q).sum()) for q in x))
        n = max(1, math.ceil(1.3 * rho * t))
        for _ in range(n):
            term = [q * (t / n) for q in force(v, True)]
            v = [q + z for q, z in zip(v, term)]
            for k in range(2, 30):
                term = [q * (t / n / k) for q in force(term, False)]
                v = [q + z for q, z in zip(v, term)]
                if k > 8 and all(float(z.abs().max()) < 1e-17 * float(q.abs().max()) for q, z in zip(v, term)
                                 if q.numel()):
                    break
        return v


def exact(case, seed):
    kind, steps = case["kind"], case["steps"]
    if kind == "sparse":
        return None  # which entries are stored follows from the round-off of every sum
    if kind == "batch":
        out = []
        for b, c in enumerate(_sub_cases(case)):
            s = seed + 1000 * b
            x = _Exact(c, s, ports=True)
            dt = _dt(x.nodes, x.tets, c["order"])
            wave = _wave(c, s, steps, dt)
            v = x.vec(_start(c, x.nodes, x.tets, c["order"], s, 0))
            out.append(x.flat(x.lserk(v, dt, steps, lambda u, k: x.apply(u, wave[k]))))
        return out
    x = _Exact(case, seed)
    dt = _dt(x.nodes, x.tets, case["order"])
    y = _start(case, x.nodes, x.tets, case["order"], seed, len(x.debye))
    v = x.vec(y)
    n_eh = x.K * x.np_ * 6
    dof = _source_dof(case, n_eh, seed)
    wave = _wave(case, seed, steps, dt) if case["drive"] == "point" else None

    def driven(u, g):
        k = x.apply(u)
        if g is not None:
            x.add_point(k, dof, float(g))
        return k

    if kind == "apply":
        return x.flat(x.apply(v))
    if kind in ("lserk", "probes"):
        at = torch.as_tensor(np.random.default_rng([seed, 5]).integers(0, n_eh, N_PROBES), device=x.D.device)
        e, r = at // (x.np_ * 6), at % (x.np_ * 6)
        rows = torch.empty(steps + 1, N_PROBES, dtype=torch.float64, device=x.D.device)

        def record(s, u):
            rows[s + 1] = u[0][r // 6, r % 6, e]

        record(-1, v)
        v = x.lserk(v, dt, steps, lambda u, s: driven(u, None if wave is None else wave[s]),
                    record if kind == "probes" else None)
        return (rows.cpu().numpy(), x.flat(v)) if kind == "probes" else x.flat(v)
    if kind == "kcl":
        rows = [y]
        for s in range(steps):
            g = None if wave is None else wave[s]
            v = x.flow(v, _horizon(case, dt), lambda u, b: driven(u, g if b else None))
            rows.append(x.flat(v))
        return np.stack(rows)
    g = 1.0 if kind == "etd" else None
    return x.flat(x.flow(v, _horizon(case, dt), lambda u, b: driven(u, g if b else None)))
