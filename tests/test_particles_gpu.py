"""Lennard-Jones and bar-and-hinge potentials on the GPU vs the reference's
golden vectors, its unit-test known answers and the oracle."""
import math

import numpy as np
import pytest

from conftest import golden
from minim_amd._capi import MinimError
from oracle_bind import OracleBaH, OracleLJ, OracleLJPBC, oracle_fire, oracle_lbfgs

pytestmark = pytest.mark.gpu

TOL = {"fp64": 1e-12, "fp32": 1e-5}


def rel_err(a, b):
    a, b = np.asarray(a, dtype=np.float64), np.asarray(b, dtype=np.float64)
    return np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300)


def r32(x):
    return np.asarray(x, dtype=np.float64).astype(np.float32).astype(np.float64)


# ---------------------------------------------------------------- Lennard-Jones
def test_lj_dimer_known_answer(gpu):
    # State_test.cpp:33-51 through every State entry point
    m = gpu
    s = m.State(m.Lj3d(), [0, 0, 0, 2, 0, 0])
    gex = [-93.0 / 512, 0, 0, 93.0 / 512, 0, 0]
    assert s.energy() == pytest.approx(-63.0 / 1024, rel=1e-15)
    np.testing.assert_allclose(s.gradient(), gex, atol=1e-15)
    e, g = s.energyGradient()
    assert e == pytest.approx(-63.0 / 1024, rel=1e-15)
    np.testing.assert_allclose(g, gex, atol=1e-15)
    assert s.energy([0, 0, 0, 2, 0, 0]) == pytest.approx(-63.0 / 1024, rel=1e-15)
    assert s.blockEnergy() == s.procEnergy() == s.allEnergy()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("case", range(3))
def test_lj_golden_vectors(gpu, case, prec):
    m = gpu
    c = golden("lj")[case]
    x = np.array(c["x"]) if prec == "fp64" else r32(c["x"])
    s = m.State(m.LjNd(c["ndim"]), x, prec)
    e, g = s.energyGradient()
    o = OracleLJ(c["ndim"], c["n"])
    eo, go = o.energy(x), o.gradient(x)
    assert abs(e - eo) <= TOL[prec] * abs(eo)
    assert rel_err(g, go) <= TOL[prec]
    if prec == "fp64":
        assert e == pytest.approx(c["energy"], rel=1e-12)
        assert rel_err(g, c["gradient"]) <= 1e-12


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 257, 1024, 1025, 2047, 2048, 2050])
@pytest.mark.parametrize("dim", [1, 2, 3, 4])
def test_lj_all_pairs_sizes(gpu, dim, n, prec):
    """Energy, gradient and the trial energy at x + t d around the kernel's
    block and group sizes, against numpy's FP64 pair sums, which add pairwise.
    (The oracle adds its n(n-1)/2 terms one after another: at n = 2,047 in one
    dimension each of the far pairs, below half an ulp of the running sum, is
    lost there -- about 2,047 * 4/5 * 185^-5 = 8e-9 of 2,010, over 1e-12.)  On a
    jittered lattice the pair terms of one sign dominate, so the rounding errors
    of the sums stay within the usual tolerance."""
    import torch

    def pair_sums(x):
        p = x.reshape(n, dim)
        dx = p[:, None, :] - p[None, :, :]
        r2 = (dx * dx).sum(-1)
        np.fill_diagonal(r2, 1.0)
        i6 = r2 ** -3
        pair, f = 4 * (i6 * i6 - i6), -24 * (2 * i6 * i6 - i6) / r2
        np.fill_diagonal(pair, 0.0)
        np.fill_diagonal(f, 0.0)
        return 0.5 * pair.sum(), np.einsum("ijk,ij->ik", dx, f).reshape(-1)

    m = gpu
    print("case lj all pairs", dim, n, prec, flush=True)
    rng = np.random.default_rng(1000 * dim + n)
    side = int(np.ceil(n ** (1.0 / dim) - 1e-9))
    pts = np.array(np.meshgrid(*[np.arange(side) * 1.15] * dim, indexing="ij")).reshape(dim, -1).T[:n]
    x = r32((pts + rng.uniform(-0.05, 0.05, pts.shape)).reshape(-1))
    d = r32(rng.uniform(-0.1, 0.1, x.shape))
    eo, go = pair_sums(x)
    h = m.LjNd(dim).handle(x)
    dt = torch.float64 if prec == "fp64" else torch.float32
    xd = torch.tensor(x, dtype=dt, device="cuda")
    dd = torch.tensor(d, dtype=dt, device="cuda")
    g = torch.full_like(xd, float("nan"))
    e = m.potential_eval(h, prec, xd.data_ptr(), x.size, g_ptr=g.data_ptr())
    g2 = torch.full_like(xd, float("nan"))
    m.potential_eval(h, prec, xd.data_ptr(), x.size, g_ptr=g2.data_ptr(), want_energy=False)
    et = m.potential_eval(h, prec, xd.data_ptr(), x.size, d_ptr=dd.data_ptr(), t=0.25)
    assert torch.equal(g, g2)
    if n == 1:
        assert e == 0.0 and et == 0.0 and not g.any()
        return
    assert abs(e - eo) <= TOL[prec] * abs(eo)
    eto = pair_sums(x + 0.25 * d)[0]
    assert abs(et - eto) <= TOL[prec] * abs(eto)
    assert rel_err(g.cpu().numpy(), go) <= TOL[prec]


def lattice(n_side, a, jitter, rng):
    g = np.arange(n_side) * a
    pts = np.array(np.meshgrid(g, g, g, indexing="ij")).reshape(3, -1).T
    return (pts + rng.uniform(-jitter, jitter, pts.shape)).reshape(-1)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("n_side", [5, 9])
def test_lj_cutoff_vs_oracle(gpu, n_side, prec):
    """Truncated-shifted LJ in a periodic box (cell list for 9^3, brute-force
    list for the small 5^3 box) vs the oracle's minimum-image all-pairs sum."""
    m = gpu
    rng = np.random.default_rng(n_side)
    a = 1.1
    L = n_side * a
    x = lattice(n_side, a, 0.15, rng)
    x = x if prec == "fp64" else r32(x)
    n = n_side ** 3
    pot = m.Lj3d().setCutoff(2.5, [L, L, L], 0.3)
    s = m.State(pot, x, prec)
    e, g = s.energyGradient()
    assert pot.listBuilds(s) == 1
    # the longest list: the most minimum-image neighbours within rc + skin
    p = x.reshape(-1, 3).astype(np.float64)
    dv = p[:, None, :] - p[None, :, :]
    dv -= L * np.rint(dv / L)
    r2 = (dv * dv).sum(-1)
    np.fill_diagonal(r2, np.inf)
    assert pot.maxNeighbours(s) == int((r2 < 2.8 ** 2).sum(1).max())
    o = OracleLJPBC(n, L, 2.5)
    assert abs(e - o.energy(x)) <= TOL[prec] * abs(o.energy(x))
    assert rel_err(g, o.gradient(x)) <= TOL[prec]
    # move particles beyond skin/2: the list must be rebuilt, results stay exact
    y = x + rng.uniform(-0.3, 0.3, x.shape)
    y = y if prec == "fp64" else r32(y)
    e2, g2 = s.energyGradient(y)
    assert pot.listBuilds(s) == 2
    assert abs(e2 - o.energy(y)) <= TOL[prec] * abs(o.energy(y))
    assert rel_err(g2, o.gradient(y)) <= TOL[prec]
    # particles far outside the box (whole periods added, different per
    # particle): the same energy and forces as their images inside it
    k = rng.integers(-4, 5, (n, 1)) * L
    z = (y.reshape(-1, 3) + k).reshape(-1)
    z = z if prec == "fp64" else r32(z)
    e3, g3 = s.energyGradient(z)
    assert abs(e3 - o.energy(z)) <= 10 * TOL[prec] * abs(o.energy(z))
    assert rel_err(g3, o.gradient(z)) <= 10 * TOL[prec]


def test_lj_fire_cluster(gpu):
    """Fire relaxes a 27-particle cluster; same minimum as the oracle's Fire."""
    m = gpu
    rng = np.random.default_rng(11)
    x0 = lattice(3, 1.12, 0.05, rng)
    s = m.State(m.Lj3d(), x0)
    f = m.Fire().setMaxIter(20000)
    f.minimise(s)
    o = OracleLJ(3, 27)
    _, so = oracle_fire(o, x0, max_iter=20000)
    assert f.stats["converged"] and so["converged"]
    assert s.energy() == pytest.approx(so["energy"], rel=1e-8)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_fire_dt0_first_step(gpu, prec):
    """Fire with an initial time step: iteration 0 has v = 0, so p = 0, v = -dt0 g
    and dt halves before the step (Fire.cpp:50-67): x1 = x0 - 0.5 dt0^2 g(x0)."""
    m = gpu
    rng = np.random.default_rng(5)
    n_side, a = 5, 1.1
    L = n_side * a
    x0 = lattice(n_side, a, 0.1, rng)
    x0 = x0 if prec == "fp64" else r32(x0)
    pot = m.Lj3d().setCutoff(2.5, [L, L, L], 0.3)
    s = m.State(pot, x0, prec)
    g0 = s.gradient()
    f = m.Fire(0.02).setDt0(0.002).setMaxIter(0)
    x1 = f.minimise(s)
    np.testing.assert_allclose(x1, x0 - 0.5 * 0.002 ** 2 * g0, rtol=TOL[prec], atol=TOL[prec] * np.abs(x0).max())


def test_fire_max_force_lj_cutoff_vs_oracle(gpu):
    """The LJ benchmark's minimiser settings on a small periodic box: Fire with
    dt0 0.002, dtMax 0.02, no line search, converged when the largest
    per-particle force is below 1e-6; same minimum as the oracle's Fire on the
    minimum-image all-pairs potential."""
    m = gpu
    rng = np.random.default_rng(31)
    n_side, a = 6, (1 / 0.85) ** (1 / 3)  # density 0.85
    L = n_side * a
    x0 = lattice(n_side, a, 0.08, rng)
    n = n_side ** 3
    pot = m.Lj3d().setCutoff(2.5, [L, L, L], 0.3)
    s = m.State(pot, x0)
    s.convergence = 1e-6
    f = m.Fire(0.02).setDt0(0.002).setMaxForceConvergence(3).setMaxIter(50000)
    x = f.minimise(s)
    o = OracleLJPBC(n, L, 2.5)
    xo, so = oracle_fire(o, x0, dt_max=0.02, dt0=0.002, max_force_dim=3, max_iter=50000, linesearch="none",
                         convergence=1e-6)
    print(f.stats, so, flush=True)
    assert f.stats["converged"] and so["converged"]
    assert f.stats["grad_max"] < 1e-6
    gmax = np.sqrt((o.gradient(x).reshape(-1, 3) ** 2).sum(axis=1)).max()
    assert gmax < 2e-6
    assert s.energy() == pytest.approx(so["energy"], rel=1e-8)
    assert abs(f.stats["iterations"] - so["iterations"]) <= max(20, 0.2 * so["iterations"])


# ---------------------------------------------------------------- BarAndHinge
def bah_from_case(m, c, use_tri=False):
    p = m.BarAndHinge()
    if use_tri:
        p.setTriangulation(c["tri"]).setRigidity(c["kb"], c["kh"])
        if c["l0"] is not None:
            p.setLength0(c["l0"])
        if c["t0"] is not None:
            p.setTheta0(c["t0"])
    else:
        p.setBondList(c["bars"]).setHingeList(c["hinges"]).setRigidity(c["bar_k"], c["hinge_k"])
        p.setLength0(c["bar_l0"]).setTheta0(c["hinge_t0"])
    if c["force"] is not None:
        p.setForce(c["force"])
    if c["fixed"]:
        p.setConstraints(c["fixed"])
    return p


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("case", range(2))
def test_bah_golden_vectors(gpu, case, prec):
    m = gpu
    c = golden("bah")[case]
    x = np.array(c["x"]) if prec == "fp64" else r32(c["x"])
    s = m.State(bah_from_case(m, c), c["x0"], prec)
    e, g = s.energyGradient(x)
    nnode = len(x) // 3
    fixed = None
    if c["fixed"]:
        fixed = np.zeros(3 * nnode, np.uint8)
        fixed[c["fixed"]] = 1
    o = OracleBaH(nnode, c["bars"], c["bar_k"], c["bar_l0"], c["hinges"], c["hinge_k"], c["hinge_t0"],
                  force=None if c["force"] is None else np.array(c["force"]), fixed=fixed)
    eo, go = o.energy(x), o.gradient(x)
    assert abs(e - eo) <= TOL[prec] * abs(eo)
    assert rel_err(g, go) <= TOL[prec]
    if prec == "fp64":
        assert e == pytest.approx(c["energy"], rel=1e-12)
        assert rel_err(g, c["gradient"]) <= 1e-12
        if c["fixed"]:
            assert np.all(g[c["fixed"]] == 0)
        # the same sheet built from its triangulation (O(T) list construction)
        s2 = m.State(bah_from_case(m, c, use_tri=True), c["x0"], prec)
        e2, g2 = s2.energyGradient(x)
        assert e2 == pytest.approx(e, rel=1e-14)
        assert rel_err(g2, g) <= 1e-14


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("nnode", [8, 121, 700])
def test_bah_any_lists_vs_oracle(gpu, nnode, prec):
    """Bond and hinge lists that are no sheet, with their own parameters, a
    force per node and single fixed components: every hinge at one hub (more
    than a chunk of the kernel holds for 700 nodes), bars between any two
    nodes.  The nodes lie on a unit sphere around the hub, and a hinge's
    triangles have a sine of at least 0.7 at the hub, so that an element's
    rounding stays within a few tens of its operands': TOL."""
    import torch

    m = gpu
    print("case bah lists", nnode, prec, flush=True)
    rng = np.random.default_rng(nnode)
    p = rng.normal(size=(nnode, 3))
    p /= np.linalg.norm(p, axis=1)[:, None]
    hub = nnode // 3
    p[hub] = 0
    bars, hinges = [], []
    for _ in range(3 * nnode):
        a, b = rng.integers(nnode, size=2)
        if a != b and np.linalg.norm(p[a] - p[b]) > 0.3:
            bars.append((a, b))
    for _ in range(40 * nnode):
        i, j, k = rng.integers(nnode, size=3)
        if hub not in (i, j, k) and len({i, j, k}) == 3 and max(abs(p[i] @ p[j]), abs(p[j] @ p[k])) < 0.7:
            hinges.append((i, hub, j, k))
    if nnode == 700:
        assert len(hinges) > 4 * 480
    nb, nh = len(bars), len(hinges)
    bk, bl = rng.uniform(0.5, 2, nb), rng.uniform(0.5, 1, nb)
    hk, ht = rng.uniform(0.5, 2, nh), rng.uniform(2, 4, nh)
    force = rng.normal(size=3 * nnode)
    fixed = rng.choice(3 * nnode, nnode // 2, replace=False)
    x = p.reshape(-1)
    x = r32(x) if prec == "fp32" else x
    pot = m.BarAndHinge().setForce(force.tolist())
    assert nb and nh
    pot.setBondList(np.array(bars)).setHingeList(np.array(hinges)).setRigidity(bk, hk).setLength0(bl).setTheta0(ht)
    pot.setConstraints(fixed.tolist())
    fx = np.zeros(3 * nnode, np.uint8)
    fx[fixed] = 1
    o = OracleBaH(nnode, np.array(bars), bk, bl, np.array(hinges), hk, ht, force=force, force_per_node=True, fixed=fx)
    s = m.State(pot, x, prec)
    e, g = s.energyGradient(x)
    eo, go = o.energy(x), o.gradient(x)
    scale = np.sum(bk) + np.sum(hk) + np.sum(np.abs(force))  # the energy's terms have either sign
    assert abs(e - eo) <= TOL[prec] * max(abs(eo), scale)
    assert rel_err(g, go) <= TOL[prec]
    assert np.all(g[fixed] == 0)
    assert np.array_equal(s.gradient(x), g)
    assert s.energy(x) == e
    # the step: into a buffer of its own, and over its input
    h = pot.handle(x)
    dt = torch.float64 if prec == "fp64" else torch.float32
    d = torch.tensor(rng.normal(0, 0.01, x.size), dtype=dt, device="cuda")
    out = []
    for over in (False, True):
        xd = torch.tensor(x, dtype=dt, device="cuda")
        xo = xd if over else torch.empty_like(xd)
        gd = torch.empty_like(xd)
        es = m.potential_eval_step(h, prec, prec, xd.data_ptr(), x.size, d.data_ptr(), 0.5, xo.data_ptr(), gd.data_ptr())
        out.append((es, xo.cpu(), gd.cpu()))
    assert out[0][0] == out[1][0]
    assert torch.equal(out[0][1], out[1][1]) and torch.equal(out[0][2], out[1][2])


def test_bah_two_triangle_minima(gpu):
    # BarAndHinge_test.cpp:13-56: L-BFGS minima for five rest angles, within 1e-4
    m = gpu
    c = golden("bah")[2]
    dz = math.sqrt(2) / 2
    s2 = math.sqrt(2)
    expected = [[0, 0, 0.5 + dz, 0, -s2, 0.5 - dz, 0, s2, 0.5 - dz, 0, 0, 0.5 + dz],
                [-1, 0, 1, 0, -s2, 0, 0, s2, 0, 1, 0, 1],
                [-s2, 0, 0.5, 0, -s2, 0.5, 0, s2, 0.5, s2, 0, 0.5],
                [-1, 0, 0, 0, -s2, 1, 0, s2, 1, 1, 0, 0],
                [0, 0, 0.5 - dz, 0, -s2, 0.5 + dz, 0, s2, 0.5 + dz, 0, 0, 0.5 - dz]]
    for mn_ref, ex in zip(c["minima"], expected):
        p = m.BarAndHinge().setTriangulation(c["tri"]).setRigidity(c["kb"], c["kh"]).setTheta0(mn_ref["theta0"])
        s = m.State(p, c["x0"])
        x = m.Lbfgs().minimise(s)
        np.testing.assert_allclose(x, ex, atol=1e-4)
        np.testing.assert_allclose(x, mn_ref["x"], atol=1e-6)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_bah_sheet_vs_oracle(gpu, prec):
    """The benchmark sheet's construction at 256^2 nodes (equilateral lattice
    compressed by 0.95, clamped x edges, z noise): energy and gradient at the
    start and at a perturbed point against the oracle, for the energy pass
    that stores the hinge angles, the gradient-only pass and a trial point."""
    import torch
    from bench import sheet_triangles

    m = gpu
    nside = 256
    tri = sheet_triangles(nside, nside)
    i, j = np.meshgrid(np.arange(nside), np.arange(nside), indexing="ij")
    rng = np.random.default_rng(78)
    x0 = np.stack([0.95 * (i - 0.5 * j), (np.sqrt(3) / 2) * j, rng.normal(0, 0.01, i.shape)], -1).reshape(-1)
    edge = np.where((i == 0) | (i == nside - 1), 1, 0).reshape(-1).nonzero()[0]
    fixed = np.stack([3 * edge, 3 * edge + 1, 3 * edge + 2], 1).reshape(-1)
    pot = m.BarAndHinge().setTriangulation(tri).setRigidity(1.0, 0.01).setLength0(1.0).setTheta0(np.pi)
    pot.setConstraints(fixed.tolist())
    bonds, hinges = m.triangulation_lists(tri)
    nnode = nside * nside
    fx = np.zeros(3 * nnode, np.uint8)
    fx[fixed] = 1
    o = OracleBaH(nnode, bonds, np.ones(len(bonds)), np.ones(len(bonds)), hinges, np.full(len(hinges), 0.01),
                  np.full(len(hinges), np.pi), fixed=fx)
    x1 = x0 + rng.normal(0, 0.02, x0.size)
    xs = r32(x1) if prec == "fp32" else x1
    s = m.State(pot, x0, prec)
    e, g = s.energyGradient(xs)
    eo, go = o.energy(xs), o.gradient(xs)
    assert abs(e - eo) <= TOL[prec] * abs(eo)
    assert rel_err(g, go) <= TOL[prec]
    assert np.all(g[fixed] == 0)
    assert rel_err(s.gradient(xs), go) <= TOL[prec]
    # energy at a trial point x + t*d (materialised before the energy pass)
    h = pot.handle(x0)
    dt = torch.float64 if prec == "fp64" else torch.float32
    xd = torch.tensor(xs, dtype=dt, device="cuda")
    d = torch.tensor(rng.normal(0, 0.01, x0.size), dtype=dt, device="cuda")
    t = 0.625
    et = m.potential_eval(h, prec, xd.data_ptr(), x0.size, d_ptr=d.data_ptr(), t=t)
    xt = (xd + torch.tensor(t, dtype=dt, device="cuda") * d).double().cpu().numpy()
    assert abs(et - o.energy(xt)) <= TOL[prec] * abs(o.energy(xt))


@pytest.mark.parametrize("prec", ["fp64", "fp32", "mixed"])
def test_bah_fused_step_matches_separate_passes(gpu, prec):
    """The L-BFGS line search's fused accepted step for the bar-and-hinge
    sheet (x + t*d written out, then energy and gradient there in one energy
    pass and the gather) gives bit for bit the trial energy of the separate
    trial pass, and the gradient pass at the point it wrote; fixed DOFs stay
    zero."""
    import torch
    from bench import sheet_triangles

    m = gpu
    nside = 40
    print("case bah fused step", nside, prec, flush=True)
    tri = sheet_triangles(nside, nside)
    i, j = np.meshgrid(np.arange(nside), np.arange(nside), indexing="ij")
    rng = np.random.default_rng(81)
    x0 = np.stack([0.95 * (i - 0.5 * j), (np.sqrt(3) / 2) * j, rng.normal(0, 0.01, i.shape)], -1).reshape(-1)
    edge = np.where((i == 0) | (i == nside - 1), 1, 0).reshape(-1).nonzero()[0]
    fixed = np.stack([3 * edge, 3 * edge + 1, 3 * edge + 2], 1).reshape(-1)
    pot = m.BarAndHinge().setTriangulation(tri).setRigidity(1.0, 0.01).setLength0(1.0).setTheta0(np.pi)
    pot.setConstraints(fixed.tolist())
    n = x0.size
    h = pot.handle(x0)
    px = "fp32" if prec == "fp32" else "fp64"
    pv = "fp64" if prec == "fp64" else "fp32"
    tx = torch.float32 if px == "fp32" else torch.float64
    tv = torch.float32 if pv == "fp32" else torch.float64
    x = torch.tensor(x0 + rng.normal(0, 0.02, n), dtype=tx, device="cuda")
    d = torch.tensor(rng.normal(0, 0.01, n), dtype=tv, device="cuda")
    t = 0.625
    xo = torch.empty_like(x)
    g = torch.empty(n, dtype=tv, device="cuda")
    e = m.potential_eval_step(h, px, pv, x.data_ptr(), n, d.data_ptr(), t, xo.data_ptr(), g.data_ptr())
    gref = torch.empty(n, dtype=tv, device="cuda")
    if prec == "mixed":
        eref = m.potential_eval_mixed(h, x.data_ptr(), n, d_ptr=d.data_ptr(), t=t)
        m.potential_eval_mixed(h, xo.data_ptr(), n, g_ptr=gref.data_ptr(), want_energy=False)
    else:
        eref = m.potential_eval(h, px, x.data_ptr(), n, d_ptr=d.data_ptr(), t=t)
        m.potential_eval(h, px, xo.data_ptr(), n, g_ptr=gref.data_ptr(), want_energy=False)
    torch.cuda.synchronize()
    assert e == eref
    assert torch.equal(g, gref)
    assert torch.all(g[torch.tensor(fixed, device="cuda")] == 0)
    xt = x.double() + t * d.double()
    ulp = 2.0 ** -22 if px == "fp32" else 2.0 ** -50
    assert torch.allclose(xo.double(), xt, rtol=ulp, atol=ulp)


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
def test_bah_lbfgs_fused_step_keeps_the_trajectory(gpu, prec):
    """L-BFGS on the bar-and-hinge sheet takes its accepted first trials
    through the fused step, whose gradient follows in a pass of its own.  A maxStep too large to bind runs the same algorithm through the
    separate trial energy, axpy and gradient passes: after 300 iterations the
    coordinates, energy and evaluation counts agree bit for bit."""
    from bench import sheet_triangles

    m = gpu
    nside = 24
    print("case bah lbfgs fused trajectory", nside, prec, flush=True)
    tri = sheet_triangles(nside, nside)
    i, j = np.meshgrid(np.arange(nside), np.arange(nside), indexing="ij")
    rng = np.random.default_rng(82)
    x0 = np.stack([0.95 * (i - 0.5 * j), (np.sqrt(3) / 2) * j, rng.normal(0, 0.01, i.shape)], -1).reshape(-1)
    edge = np.where((i == 0) | (i == nside - 1), 1, 0).reshape(-1).nonzero()[0]
    fixed = np.stack([3 * edge, 3 * edge + 1, 3 * edge + 2], 1).reshape(-1)
    out = []
    for cap in (0.0, 1e30):
        p = m.BarAndHinge().setTriangulation(tri).setRigidity(1.0, 0.01).setLength0(1.0).setTheta0(np.pi)
        p.setConstraints(fixed.tolist())
        s = m.State(p, x0, "fp64")
        lb = m.Lbfgs().setM(10).setMaxIter(300).setPrecision(prec)
        if cap:
            lb.setMaxStep(cap)
        lb.minimise(s)
        st = lb.stats
        out.append((s.coords(), s.energy(), st["iterations"], st["n_energy"], st["n_gradient"]))
    assert np.array_equal(out[0][0], out[1][0])
    assert out[0][1:] == out[1][1:]


def test_bah_mixed_evaluation_and_minimisation(gpu):
    """The mixed schedule's evaluation of the bar-and-hinge sheet: FP64
    coordinates and arithmetic with FP32 direction and gradient.  The energy
    is the FP64 evaluation's bit for bit, the gradient its FP32 rounding
    (fixed DOFs zero), and a trial point x + t d with d in FP32 gives the FP64
    energy at d widened to FP64.  L-BFGS m=10 with either schedule then
    reaches the tolerance (the oracle's gradient at the coordinates left),
    with the energy the oracle's at those coordinates (1e-12)."""
    import torch
    from bench import sheet_triangles

    m = gpu
    nside = 24
    tri = sheet_triangles(nside, nside)
    i, j = np.meshgrid(np.arange(nside), np.arange(nside), indexing="ij")
    rng = np.random.default_rng(79)
    x0 = np.stack([0.95 * (i - 0.5 * j), (np.sqrt(3) / 2) * j, rng.normal(0, 0.01, i.shape)], -1).reshape(-1)
    edge = np.where((i == 0) | (i == nside - 1), 1, 0).reshape(-1).nonzero()[0]
    fixed = np.stack([3 * edge, 3 * edge + 1, 3 * edge + 2], 1).reshape(-1)

    def make():
        p = m.BarAndHinge().setTriangulation(tri).setRigidity(1.0, 0.01).setLength0(1.0).setTheta0(np.pi)
        p.setConstraints(fixed.tolist())
        return p

    pot = make()
    n = x0.size
    h = pot.handle(x0)
    x = torch.tensor(x0 + rng.normal(0, 0.02, n), dtype=torch.float64, device="cuda")
    d32 = torch.tensor(rng.normal(0, 0.01, n), dtype=torch.float32, device="cuda")
    g64 = torch.empty(n, dtype=torch.float64, device="cuda")
    g32 = torch.empty(n, dtype=torch.float32, device="cuda")
    e64 = m.potential_eval(h, "fp64", x.data_ptr(), n, g_ptr=g64.data_ptr())
    emx = m.potential_eval_mixed(h, x.data_ptr(), n, g_ptr=g32.data_ptr())
    torch.cuda.synchronize()
    assert emx == e64
    assert torch.equal(g32, g64.float())
    assert torch.all(g32[torch.tensor(fixed, device="cuda")] == 0)
    t = 0.625
    assert m.potential_eval_mixed(h, x.data_ptr(), n, d_ptr=d32.data_ptr(), t=t) == m.potential_eval(
        h, "fp64", x.data_ptr(), n, d_ptr=d32.double().data_ptr(), t=t)

    bonds, hinges = m.triangulation_lists(tri)
    fx = np.zeros(n, np.uint8)
    fx[fixed] = 1
    o = OracleBaH(nside * nside, bonds, np.ones(len(bonds)), np.ones(len(bonds)), hinges,
                  np.full(len(hinges), 0.01), np.full(len(hinges), np.pi), fixed=fx)
    out = {}
    for prec in ("fp64", "mixed"):
        s = m.State(make(), x0, "fp64")
        lb = m.Lbfgs().setM(10).setMaxIter(200000).setPrecision(prec)
        lb.minimise(s)
        st = lb.stats
        print(prec, st["iterations"], st["converged"], st["energy"], flush=True)
        assert st["converged"], (prec, st)
        xs = s.coords()
        assert abs(s.energy() - o.energy(xs)) <= 1e-12 * abs(o.energy(x0))
        g = o.gradient(xs)
        assert np.sqrt(np.mean(g * g)) < 1.0001 * s.convergence
        out[prec] = s.energy()
    # The compressed sheet buckles into a very flat minimum: at a gradient RMS
    # of 1e-6 its energy is pinned only to about 1e-5 of the initial energy,
    # and the two schedules stop at different points of that valley.
    assert abs(out["mixed"] - out["fp64"]) <= 1e-5 * abs(o.energy(x0))


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("side", [7, 20, 25, 26, 33, 41])
def test_lj_cutoff_lanes_vs_lattice_sum(gpu, side, prec):
    """Cutoff mode at particle counts on either side of each choice of lanes
    per particle, force pass (16, 8, 4, 2 and 1) and list build (16 and 8):
    energy and gradient of a jittered lattice against the FP64 sum over lattice
    shifts.  FP32: a pair keeps an absolute error of one ulp of the box per
    component, and the pair force's relative change is at most 14 times the
    distance's (r > 0.75): 14 * 2^-23 * side / 0.75 per pair, a few pairs of
    which dominate a particle."""
    import torch

    m = gpu
    print("case lj lanes", side, prec, flush=True)
    a, rc = 0.85 ** (-1 / 3), 2.5
    k = np.arange(side) * a
    x = np.stack(np.meshgrid(k, k, k, indexing="ij"), -1).reshape(-1, 3)
    x = r32((x + np.random.default_rng(side).uniform(-0.1, 0.1, x.shape)).reshape(-1))
    p = torch.tensor(x, device="cuda").reshape(side, side, side, 3)
    go, eo, L = torch.zeros_like(p), 0.0, side * a
    # a pair within the cutoff is at most three lattice steps apart along each axis
    for s in np.stack(np.meshgrid(*[range(-3, 4)] * 3), -1).reshape(-1, 3):
        if not s.any():
            continue
        dx = p - torch.roll(p, s.tolist(), (0, 1, 2))
        dx = dx - L * torch.round(dx / L)
        r2 = (dx * dx).sum(-1)
        near = r2 < rc * rc
        i6 = torch.where(near, r2, 1.0) ** -3
        eo += 0.5 * float(torch.where(near, 4 * (i6 * i6 - i6) - 4 * (rc ** -12 - rc ** -6), 0.0).sum())
        go += dx * torch.where(near, -24 * (2 * i6 * i6 - i6) / r2, 0.0)[..., None]
    xd = torch.tensor(x, dtype=torch.float64 if prec == "fp64" else torch.float32, device="cuda")
    h = m.Lj3d().setCutoff(rc, [L] * 3, 0.3).handle(x)
    g = torch.empty_like(xd)
    e = m.potential_eval(h, prec, xd.data_ptr(), xd.numel(), g_ptr=g.data_ptr())
    tol = 1e-12 if prec == "fp64" else 14 * 2.0 ** -23 * side / 0.75
    assert abs(e - eo) <= tol * abs(eo)
    assert float((g.double() - go.reshape(-1)).norm()) <= tol * float(go.norm())


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_lj_list_longer_than_its_rows(gpu, prec):
    """A system so dense that a list outgrows its rows at first (343 particles
    in a box of 6 sigma, more than 128 neighbours): the list is built again with
    longer rows and the evaluation repeated, in cell mode off (fewer than three
    cells a side) and on (a dense corner of a larger box)."""
    m = gpu
    rng = np.random.default_rng(5)
    for L, spread in ((6.0, 6.0), (12.0, 6.0)):
        k = np.arange(7)
        x = np.stack(np.meshgrid(k, k, k, indexing="ij"), -1).reshape(-1, 3) * (spread / 7)
        x = r32((x + rng.uniform(-0.02, 0.02, x.shape)).reshape(-1))
        o = OracleLJPBC(len(x) // 3, L, 2.5)
        s = m.State(m.Lj3d().setCutoff(2.5, [L] * 3, 0.3), x, prec)
        e, g = s.energyGradient(x)
        tol = 1e-12 if prec == "fp64" else 1e-4
        assert abs(e - o.energy(x)) <= tol * abs(o.energy(x)) + tol
        assert rel_err(g, o.gradient(x)) <= tol


def test_lj_list_that_does_not_fit_in_memory(gpu):
    """Lists that would take 410 GB (320,000 particles, all within the list
    radius of each other): every evaluation fails with the allocation's error,
    and the next one of another system is as good as ever."""
    m = gpu
    rng = np.random.default_rng(8)
    n, L = 320000, 10.0
    s = m.State(m.Lj3d().setCutoff(5.0, [L] * 3, 4.0), rng.uniform(0, L, 3 * n), "fp32")
    for k in range(3):
        print("evaluation", k, flush=True)
        with pytest.raises(MinimError, match="memory"):
            s.energyGradient()
    del s
    x = lattice(4, 1.1, 0.05, rng)
    o = OracleLJPBC(64, 5.0, 2.5)
    e, g = m.State(m.Lj3d().setCutoff(2.5, [5.0] * 3, 0.3), x).energyGradient()
    assert abs(e - o.energy(x)) <= 1e-12 * abs(o.energy(x))
    assert rel_err(g, o.gradient(x)) <= 1e-12


@pytest.mark.parametrize("prec,sigma,eps,x", [
    ("fp32", 1.0, 1.0, [0.0, 1.1, 1e10]),        # r^4 out of range
    ("fp64", 1.0, 1.0, [0.0, 1.1, 1e80]),
    ("fp32", 5e-7, 2.0, [0.0, 3.7e-7, 1.1e-6]),  # 1 / r^6 out of range, (sigma / r)^6 not
    ("fp32", 3e9, 0.5, [0.0, 2.7e9, 9e9]),
    ("fp32", 3.4e-10, 1.65e-21, [0.0, 3.7e-10, 8e-10]),
])
def test_lj_all_pairs_range(gpu, prec, sigma, eps, x):
    """Separations and units whose powers leave the range of the type, while
    (sigma / r)^6 and the forces stay within it."""
    m = gpu
    x = np.array(x) if prec == "fp64" else r32(x)
    s = m.State(m.LjNd(1).setSigma(sigma).setEpsilon(eps), x, prec)
    e, g = s.energyGradient()
    dx = x[:, None] - x[None, :]
    np.fill_diagonal(dx, np.inf)
    q = (sigma / dx) ** 6
    assert e == pytest.approx(2 * eps * (q * q - q).sum(), rel=TOL[prec])
    assert rel_err(g, (-24 * eps * (2 * q * q - q) / dx).sum(axis=1)) <= TOL[prec]


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_lj_cutoff_range(gpu, prec):
    """Argon in SI units with a pair at 0.02 sigma: (sigma / r)^12 / r^2 leaves
    FP32's range, the force (3e12 N) does not."""
    m = gpu
    sigma, eps, rc, L = 3.4e-10, 1.65e-21, 8.5e-10, 5e-9
    x = r32([0, 0, 0, 6.8e-12, 0, 0, 2e-9, 0, 0, 2.4e-9, 0, 0])
    s = m.State(m.Lj3d().setSigma(sigma).setEpsilon(eps).setCutoff(rc, [L] * 3, 1e-10), x, prec)
    e, g = s.energyGradient()
    r = np.array([x[3], x[9] - x[6]])
    q, qc = (sigma / r) ** 6, (sigma / rc) ** 6
    f = 24 * eps * (2 * q * q - q) / r
    assert e == pytest.approx(4 * eps * (q * q - q - (qc * qc - qc)).sum(), rel=TOL[prec])
    gx = g.reshape(-1, 3)[:, 0]
    np.testing.assert_allclose(gx, [f[0], -f[0], f[1], -f[1]], rtol=10 * TOL[prec])
    assert not g.reshape(-1, 3)[:, 1:].any()


def test_bah_step_overlaps(gpu):
    """Where the fused step's outputs may lie over its inputs it gives what it
    gives in memory of its own, and it refuses the rest, touching nothing."""
    import torch
    from bench import sheet_triangles

    m = gpu
    nside, t = 12, 0.5
    rng = np.random.default_rng(3)
    i, j = np.meshgrid(np.arange(nside), np.arange(nside), indexing="ij")
    x0 = np.stack([0.95 * (i - 0.5 * j), (np.sqrt(3) / 2) * j, rng.normal(0, 0.1, i.shape)], -1).reshape(-1)
    n = x0.size
    h = (m.BarAndHinge().setTriangulation(sheet_triangles(nside, nside)).setRigidity(1.0, 0.01).setLength0(1.0)
         .setTheta0(np.pi).handle(x0))
    v = [x0, rng.normal(0, 0.01, n)]

    def run(x, d, xo, g):  # offsets in one buffer of 6 n
        b = torch.full((6 * n,), 7.0, dtype=torch.float64, device="cuda")
        b[x:x + n] = torch.tensor(v[0])
        if d != x:
            b[d:d + n] = torch.tensor(v[1])
        before = b.clone()
        p = b.data_ptr()
        try:
            e = m.potential_eval_step(h, "fp64", "fp64", p + 8 * x, n, p + 8 * d, t, p + 8 * xo, p + 8 * g)
        except ValueError:
            assert torch.equal(b, before)
            return None
        return e, b[xo:xo + n].clone(), b[g:g + n].clone()

    def same(a, b):
        return a[0] == b[0] and torch.equal(a[1], b[1]) and torch.equal(a[2], b[2])

    want = run(0, n, 2 * n, 3 * n)
    for args in ((0, n, 0, 3 * n), (0, n, 2 * n, 0), (0, n, 2 * n, n), (0, n, 0, n), (n, 3 * n, 5 * n, n + 3)):
        assert same(run(*args), want), args
    assert same(run(0, 0, 0, 3 * n), run(0, 0, 2 * n, 3 * n))  # x = x + t x
    for args in ((0, n, n, 3 * n), (0, n, n - 3, 3 * n), (0, n, 2 * n, 2 * n), (0, n, 2 * n, 3 * n - 3),
                 (0, 4 * n, 3, 2 * n), (3, 4 * n, 0, 2 * n)):
        assert run(*args) is None, args


def fire_replay(m, h, prec, x, steps, dt0, dt_max):
    """FIRE without line search (Fire.cpp:41-84) in torch around potential_eval's
    gradients: coordinates and gradient after the steps."""
    import torch

    g = torch.empty_like(x)

    def gradient():
        m.potential_eval(h, prec, x.data_ptr(), x.numel(), g_ptr=g.data_ptr(), want_energy=False)
        torch.cuda.synchronize()

    def dot(a, b):
        return float((a.double() * b.double()).sum())

    v, a, dt, n = torch.zeros_like(x), 0.1, dt0, 0
    gradient()
    for _ in range(steps):
        p = -dot(v, g)
        if p > 0:
            v = (1 - a) * v - (a * math.sqrt(dot(v, v)) / math.sqrt(dot(g, g)) + dt) * g
            n += 1
            if n > 5:
                a, dt = a * 0.99, min(dt * 1.1, dt_max)
        else:
            v = -dt * g
            n, a, dt = 0, 0.1, dt * 0.5
        x += dt * v
        gradient()
    return x, g


# sides: 16 lanes per particle in the force pass and the list build, 4 and 8, 1 and 8
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("side,dim", [(9, 3), (9, 0), (26, 3), (41, 0)])
def test_fused_fire_vs_replay(gpu, side, dim, prec):
    """Forty fused steps with a skin that forces cell-list rebuilds against the
    replay: the gradients are the same kernels' and the sums differ in order
    only, so the steps' factors agree to a few units in the last place of their
    type; forty steps of the crystal amplify that by less than 1e3."""
    import torch

    m = gpu
    print("case fused fire", side, dim, prec, flush=True)
    a, steps = 0.85 ** (-1 / 3), 40
    x0 = r32(lattice(side, a, 0.12, np.random.default_rng(side)))
    dt = torch.float64 if prec == "fp64" else torch.float32
    pot = m.Lj3d().setCutoff(2.5, [side * a] * 3, 0.1)
    s = m.State(pot, x0, prec)
    s.convergence = 1e-30
    f = m.Fire(0.02).setDt0(0.004).setMaxIter(steps - 1)
    if dim:
        f.setMaxForceConvergence(dim)
    x = f.minimise(s)
    assert pot.listBuilds(s) >= 3
    xr, gr = fire_replay(m, pot.handle(x0), prec, torch.tensor(x0, dtype=dt, device="cuda"), steps, 0.004, 0.02)
    xr, gr = xr.double().cpu().numpy(), gr.double().cpu().numpy()
    tol = 1e3 * (2.0 ** -52 if prec == "fp64" else 2.0 ** -23)
    assert np.linalg.norm(x - xr) <= tol * np.linalg.norm(xr - x0)
    assert f.stats["grad_rms"] == pytest.approx(math.sqrt((gr * gr).mean()), rel=tol)
    if dim:
        assert f.stats["grad_max"] == pytest.approx(np.linalg.norm(gr.reshape(-1, 3), axis=1).max(), rel=tol)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("L", [11.0, 12.0])
def test_fused_fire_list_outgrows_its_rows(gpu, L, prec):
    """A stretched crystal of 343 particles that contracts: lists of at most 122
    entries at first (rows hold 128), over 128 when one is built again under
    way, in brute-force (L = 11, fewer than three cells a side) and cell mode."""
    import torch

    m = gpu
    print("case fused fire rows", L, prec, flush=True)
    a, rc, skin, steps = 1.25, 3.675, 0.2, 80
    x0 = r32(lattice(7, a, 0.005, np.random.default_rng(5)))
    p = x0.reshape(-1, 3)
    d = p[:, None] - p[None]
    d -= L * np.rint(d / L)
    assert ((d * d).sum(-1) < (rc + skin) ** 2).sum(1).max() - 1 <= 128
    dt = torch.float64 if prec == "fp64" else torch.float32
    pot = m.Lj3d().setCutoff(rc, [L] * 3, skin)
    s = m.State(pot, x0, prec)
    s.convergence = 1e-30
    x = m.Fire(0.02).setDt0(0.01).setMaxIter(steps - 1).minimise(s)
    assert pot.maxNeighbours(s) > 128
    xr, _ = fire_replay(m, pot.handle(x0), prec, torch.tensor(x0, dtype=dt, device="cuda"), steps, 0.01, 0.02)
    xr = xr.double().cpu().numpy()
    tol = 1e3 * (2.0 ** -52 if prec == "fp64" else 2.0 ** -23)
    assert np.linalg.norm(x - xr) <= tol * np.linalg.norm(xr - x0)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_lj_crowded_cell_vs_oracle(gpu, prec):
    """A thousand particles in one cell of the list build (a wavefront sorts
    it), two thirds of a sigma and less apart."""
    m = gpu
    print("case lj crowded cell", prec, flush=True)
    k = np.arange(10) * 0.28 + 0.1
    x = np.stack(np.meshgrid(k, k, k, indexing="ij"), -1).reshape(-1, 3)
    rng = np.random.default_rng(12)
    x = r32((x + rng.uniform(-0.01, 0.01, x.shape))[rng.permutation(1000)].reshape(-1))
    o = OracleLJPBC(1000, 12.0, 2.5)
    e, g = m.State(m.Lj3d().setCutoff(2.5, [12.0] * 3, 0.3), x, prec).energyGradient()
    tol = 1e-12 if prec == "fp64" else 1e-4  # 14 ulp of 3 over 0.26 in a pair's force
    assert abs(e - o.energy(x)) <= tol * abs(o.energy(x))
    assert rel_err(g, o.gradient(x)) <= tol


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_lj_diverged_particles_are_no_neighbours(gpu, prec):
    """Particles at NaN and infinity when the list is built: nobody's
    neighbours, wherever they are filed, and the rest as if they were not there."""
    m = gpu
    print("case lj diverged", prec, flush=True)
    side, a = 20, 0.85 ** (-1 / 3)
    rng = np.random.default_rng(9)
    x = r32(lattice(side, a, 0.1, rng)).reshape(-1, 3)
    lost = rng.permutation(side ** 3)[:5000]
    y = x.copy()
    y[lost[:3000], rng.integers(0, 3, 3000)] = np.nan
    y[lost[3000:], rng.integers(0, 3, 2000)] = np.inf
    kept = np.setdiff1d(np.arange(side ** 3), lost)
    pot = m.Lj3d().setCutoff(2.5, [side * a] * 3, 0.3)
    e, g = m.State(pot, y.reshape(-1), prec).energyGradient()
    e0, g0 = m.State(pot, x[kept].reshape(-1), prec).energyGradient()
    tol = 1e-12 if prec == "fp64" else 1e-5  # lists in another order
    assert abs(e - e0) <= tol * abs(e0)
    assert rel_err(g.reshape(-1, 3)[kept], g0.reshape(-1, 3)) <= tol
    assert not g.reshape(-1, 3)[lost].any()
