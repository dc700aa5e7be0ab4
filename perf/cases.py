"""Performance cases of the energy+gradient and minimiser path.

Each case is one thing a program built on this framework does over and over,
through the public Python mirror of the State / Potential / Minimiser API and
the device-pointer entry points of the C ABI:

  field     PhaseField evaluation on device vectors: energy and gradient at x
            ("eg"), or the line search's trial energy at x + t d ("trial")
  pillars   the same with solid nodes, a pressure and a fixed fluid (the
            general kernel; a pillar array on a base)
  elements  PhaseFieldUnstructured: the element form of the field
  cluster   LjNd, every pair (the reference's potential)
  liquid    LjNd with a cutoff in a periodic box
  sheet     BarAndHinge on a triangulated sheet with two clamped edges
  relax     L-BFGS on one field from its initial coordinates, a fixed number
            of iterations
  fire      FIRE on the periodic liquid, a fixed number of iterations
  batch     L-BFGS on many independent two-dimensional fields in one call

The sizes are those of the benchmark and the tests, and generic ragged ones.
The minimisations stop after a few iterations so that what comes back (the
coordinates) can be compared: L-BFGS amplifies rounding differences by an
order of magnitude every few iterations.
"""
import math

import numpy as np
import torch

import minim_amd as m

SIGMA = [1.0, 0.8, 1.2]  # pairwise surface tensions of the three-fluid fields
DENSITY = 0.85           # reduced density of the liquid
RCUT = 2.5
LATTICE = (1.0 / DENSITY) ** (1.0 / 3.0)


# ------------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest call: one evaluation of the two-dimensional binary field
        # that the reference runs on a CPU; launches and latency count
        dict(name="field_128sq_fp64", kind="field", nx=128, ny=128, nz=1, nf=1, prec="fp64", op="eg"),
        # the headline: one evaluation of the largest field in the mixed
        # schedule's storage precision
        dict(name="field_256cubed_fp32", kind="field", nx=256, ny=256, nz=256, nf=3, prec="fp32", op="eg"),
        # the line search's trial energy on an ordinary, ragged field
        dict(name="trial_ragged_fp64", kind="field", nx=150, ny=131, nz=97, nf=3, prec="fp64", op="trial"),
        # droplets on a pillar array: solid nodes, pressure, a fixed fluid
        dict(name="pillars_ragged_fp64", kind="pillars", nx=160, ny=150, nz=141, prec="fp64"),
        # the element form of the three-fluid field
        dict(name="elements_fp64", kind="elements", nx=128, ny=112, nz=120, nf=3, prec="fp64"),
        # a Lennard-Jones cluster as the reference evaluates it, all pairs
        dict(name="cluster_1000_fp64", kind="cluster", n=1000, dim=3, prec="fp64"),
        # the benchmark's liquid: 64^3 particles within a cutoff
        dict(name="liquid_64cubed_fp32", kind="liquid", side=64, skin=0.3, prec="fp32"),
        # the benchmark's elastic sheet: 1024 x 1024 nodes
        dict(name="sheet_1024sq_fp64", kind="sheet", nx=1024, ny=1024, prec="fp64"),
        # the start of the headline minimisation, mixed schedule, on the device
        dict(name="relax_256cubed_mixed", kind="relax", nx=256, ny=256, nz=256, nf=3, mode="mixed", iters=8,
             host=False),
        # a small minimisation with coordinates coming from and going to the host
        dict(name="relax_128sq_fp64", kind="relax", nx=128, ny=128, nz=1, nf=1, mode="fp64", iters=30, host=True),
        # FIRE steps of a medium liquid: two dozen dependent launches and a
        # list check per step
        dict(name="fire_32cubed_fp64", kind="fire", side=32, skin=0.3, prec="fp64", iters=100),
        # a batch of uneven fields, sides spread over [32, 512]
        dict(name="batch_64_fp64", kind="batch", count=64, sides=4040, mode="fp64", iters=30),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, hi, flat):
    """Three sides of about a log-uniform number of sites in [lo, hi]."""
    n = _log(rng, lo, hi)
    if flat:
        a = math.sqrt(n) * rng.uniform(0.8, 1.25)
        return max(8, int(a)), max(8, int(n / a)), 1
    a = n ** (1 / 3) * rng.uniform(0.8, 1.2)
    b = n ** (1 / 3) * rng.uniform(0.8, 1.2)
    return max(8, int(a)), max(8, int(b)), max(8, int(n / (a * b)))


def draw(rng):
    kind = rng.choice(["field", "field", "pillars", "elements", "cluster", "liquid", "sheet", "relax", "fire", "batch"])
    prec = rng.choice(["fp64", "fp32"])
    if kind == "field":
        nf = rng.choice([1, 1, 2, 3, 3])
        nx, ny, nz = _grid(rng, 16384, 12000000 // nf, rng.random() < 0.3)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, nf=nf, prec=prec, op=rng.choice(["eg", "trial"]))
    if kind == "pillars":
        nx, ny, nz = _grid(rng, 24 ** 3, 3500000, False)
        return dict(kind=kind, nx=max(nx, 20), ny=max(ny, 20), nz=max(nz, 20), prec=prec)
    if kind == "elements":
        nx, ny, nz = _grid(rng, 4096, 1700000, rng.random() < 0.2)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, nf=rng.choice([1, 2, 3]), prec=prec)
    if kind == "cluster":
        return dict(kind=kind, n=_log(rng, 64, 4096), dim=rng.choice([2, 3]), prec=prec)
    if kind == "liquid":
        return dict(kind=kind, side=_log(rng, 9, 64), skin=round(rng.uniform(0.2, 0.4), 3), prec=prec)
    if kind == "sheet":
        return dict(kind=kind, nx=_log(rng, 24, 700), ny=_log(rng, 24, 700), prec=prec)
    if kind == "relax":
        nf = rng.choice([1, 3])
        flat = rng.random() < 0.5
        nx, ny, nz = _grid(rng, 16384, 1 << 20 if flat else 3000000, flat)
        mode = rng.choice(["fp64", "mixed"])
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, nf=nf, mode=mode, iters=8 if mode == "mixed" else 30,
                    host=flat and rng.random() < 0.5)
    if kind == "fire":
        return dict(kind=kind, side=_log(rng, 9, 40), skin=round(rng.uniform(0.2, 0.4), 3), prec="fp64",
                    iters=rng.randint(60, 100))
    return dict(kind="batch", count=_log(rng, 8, 64), sides=rng.randrange(1 << 20), mode="fp64", iters=30)


# ------------------------------------------------------------------- the inputs
_DT = {"fp64": torch.float64, "fp32": torch.float32}


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _uniform(gen, shape, lo, hi, dtype):
    """Values of dtype's own grid, so that they are the same in FP32 and FP64."""
    u = torch.rand(shape, generator=gen, device="cuda", dtype=torch.float32)
    return (lo + (hi - lo) * u).to(dtype)


def _field_input(case, gen, dtype):
    """Random initial concentrations: phi ~ U[-0.1, 0.1] for a binary field,
    uniform and renormalised to sum to one per site otherwise."""
    n, nf = case["nx"] * case["ny"] * case["nz"], case.get("nf", 3)
    if nf == 1:
        return _uniform(gen, (n, 1), -0.1, 0.1, dtype)
    u = _uniform(gen, (n, nf), 0.0, 1.0, torch.float32)
    return (u / u.sum(1, keepdim=True)).to(dtype)


def _pillar_solid(case):
    """Solid for y < ny/16 and in square pillars of a quarter of the period's
    side on a period of half the grid, up to half height."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    x = torch.arange(nx, device="cuda")[:, None, None]
    y = torch.arange(ny, device="cuda")[None, :, None]
    z = torch.arange(nz, device="cuda")[None, None, :]
    pillar = ((x % (nx // 2)) < nx // 4) & ((z % (nz // 2)) < nz // 4) & (y < ny // 2)
    return pillar | ((y < max(1, ny // 16)) & (x >= 0) & (z >= 0))


def _pillar_input(case, gen, dtype):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    solid = _pillar_solid(case)
    liquid = (torch.arange(ny, device="cuda")[None, :, None] > 3 * ny // 4).expand(nx, ny, nz) & ~solid
    c = torch.stack([solid, liquid, ~solid & ~liquid], -1).reshape(-1, 3).to(torch.float32)
    noise = _uniform(gen, c.shape, -0.02, 0.02, torch.float32)
    return (c + noise * (~solid).reshape(-1, 1)).to(dtype)


def _cluster_input(case, gen, dtype):
    side = math.ceil(case["n"] ** (1 / case["dim"]) - 1e-9)
    grid = torch.meshgrid(*[torch.arange(side, device="cuda", dtype=torch.float32) * 1.12] * case["dim"], indexing="ij")
    x = torch.stack(grid, -1).reshape(-1, case["dim"])[:case["n"]]
    return (x + _uniform(gen, x.shape, -0.05, 0.05, torch.float32)).to(dtype)


def _liquid_input(case, gen, dtype):
    """A simple cubic lattice jittered by U[-0.1, 0.1]."""
    s = case["side"]
    grid = torch.meshgrid(*[torch.arange(s, device="cuda", dtype=torch.float32) * LATTICE] * 3, indexing="ij")
    x = torch.stack(grid, -1).reshape(-1, 3)
    return (x + _uniform(gen, x.shape, -0.1, 0.1, torch.float32)).to(dtype)


def _sheet_input(case, gen, dtype):
    """An equilateral lattice compressed by 5 % along x with out-of-plane
    noise of 0.01."""
    i, j = torch.meshgrid(torch.arange(case["nx"], device="cuda", dtype=torch.float32),
                          torch.arange(case["ny"], device="cuda", dtype=torch.float32), indexing="ij")
    z = 0.01 * torch.randn(i.shape, generator=gen, device="cuda", dtype=torch.float32)
    return torch.stack([0.95 * (i - 0.5 * j), math.sqrt(3) / 2 * j, z], -1).reshape(-1, 3).to(dtype)


def _sheet_triangles(nx, ny):
    i, j = np.meshgrid(np.arange(nx - 1), np.arange(ny - 1), indexing="ij")
    a = (i * ny + j).reshape(-1)
    b, c, d = a + ny, a + ny + 1, a + 1
    return np.stack([np.stack([a, b, c], 1), np.stack([a, c, d], 1)], 1).reshape(-1, 3).astype(np.int32)


def _sheet_clamped(nx, ny):
    """The nodes of the two x edges."""
    return np.concatenate([np.arange(ny), (nx - 1) * ny + np.arange(ny)])


def _batch_sides(case):
    """Sides log-uniform in [32, 512], set by the case."""
    u = np.random.default_rng(case["sides"]).uniform(size=case["count"])
    return [int(s) for s in np.exp(np.log(32) + u * (np.log(512) - np.log(32)))]


def _batch_instances(case, gen):
    """Interface widths in [1, 3] and fields in [-0.1, 0.1], from the generator."""
    sides = _batch_sides(case)
    u = torch.rand(case["count"], generator=gen, device="cuda", dtype=torch.float64).cpu().numpy()
    xs = [_uniform(gen, (s * s,), -0.1, 0.1, torch.float64) for s in sides]
    return sides, [float(w) for w in 1.0 + 2.0 * u], xs


def _phase_field(case, cls=None):
    nf = case.get("nf", 3)
    p = (cls or m.PhaseField)().setNFluid(nf).setGridSize([case["nx"], case["ny"], case["nz"]])
    p.setSurfaceTension(SIGMA if nf == 3 else 1.0).setInterfaceSize(1.0 if nf == 1 else 2.0)
    if case["kind"] == "pillars":
        p.setSolid(_pillar_solid(case).reshape(-1).cpu().numpy()).setFixFluid(0).setPressure([0.0, 0.05, 0.0])
    return p


def _host(x):
    return x.detach().to(torch.float64).reshape(-1).cpu().numpy()


def prepare(case, seed):
    kind, gen = case["kind"], _gen(seed)
    prec = case.get("prec", "fp64")
    dtype = _DT[prec]
    st = dict(case=case, prec=prec)
    if kind in ("field", "pillars", "elements", "cluster", "liquid", "sheet"):
        # an evaluation: the initialised potential and device buffers
        make = dict(field=_field_input, pillars=_pillar_input, elements=_field_input, cluster=_cluster_input,
                    liquid=_liquid_input, sheet=_sheet_input)[kind]
        x = make(case, gen, dtype).contiguous()
        if kind == "cluster":
            pot = m.LjNd(case["dim"])
        elif kind == "liquid":
            pot = m.Lj3d().setCutoff(RCUT, [case["side"] * LATTICE] * 3, case["skin"])
        elif kind == "sheet":
            nx, ny = case["nx"], case["ny"]
            pot = m.BarAndHinge().setTriangulation(_sheet_triangles(nx, ny)).setRigidity(1.0, 0.01)
            pot.setLength0(1.0).setTheta0(math.pi)
            edge = _sheet_clamped(nx, ny)
            pot.setConstraints(np.stack([3 * edge, 3 * edge + 1, 3 * edge + 2], 1).reshape(-1).tolist())
        else:
            pot = _phase_field(case, m.PhaseFieldUnstructured if kind == "elements" else None)
        st.update(handle=pot.handle(_host(x)), x=x, e=torch.zeros(1, dtype=torch.float64, device="cuda"))
        if case.get("op") == "trial":
            st["d"] = _uniform(gen, x.shape, -0.05, 0.05, dtype)
        else:
            st["g"] = torch.empty_like(x)
        return st
    if kind == "relax":
        x = _field_input(case, gen, torch.float32).to(torch.float64)
        host = _host(x)
        st.update(state=m.State(_phase_field(case), host),
                  mini=m.Lbfgs().setM(5).setMaxIter(case["iters"] - 1).setPrecision(case["mode"]))
        if case["host"]:
            st["x0"] = host
        else:
            st["x0"] = x.reshape(-1)
            if case["mode"] == "mixed":
                st["state"].setPrecision("fp32")
                st["x0"] = st["x0"].to(torch.float32)
        return st
    if kind == "fire":
        x = _liquid_input(case, gen, torch.float32).to(dtype)
        pot = m.Lj3d().setCutoff(RCUT, [case["side"] * LATTICE] * 3, case["skin"])
        st.update(state=m.State(pot, _host(x), prec), x0=x.reshape(-1),
                  mini=m.Fire(0.02).setDt0(0.002).setMaxForceConvergence(3).setMaxIter(case["iters"] - 1))
        return st
    sides, widths, xs = _batch_instances(case, gen)
    states = []
    for s, w, x in zip(sides, widths, xs):
        pf = m.PhaseField().setNFluid(1).setGridSize([s, s, 1]).setSurfaceTension(1.0).setInterfaceSize(w)
        states.append(m.State(pf, _host(x)))
    st.update(states=states, x0=xs, mini=m.Lbfgs().setM(5).setMaxIter(case["iters"] - 1).setPrecision(case["mode"]))
    return st


# ------------------------------------------------------------------- one pass
class _DeviceArray:
    """A State's device coordinates as an array that torch can wrap."""

    def __init__(self, ptr, n, prec):
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=(n,), version=3, strides=None,
                                             typestr="<f8" if prec == "fp64" else "<f4")


def _coords(state):
    return torch.as_tensor(_DeviceArray(state.device_coords(), state.ndof, state.precision), device="cuda")


def _set_coords(state, x0):
    """New device coordinates for a State, without a trip through the host."""
    _coords(state).copy_(x0)
    m._capi.check(m.lib.minim_state_mark_coords_changed(state.ptr))


def run(st):
    case, kind = st["case"], st["case"]["kind"]
    stream = torch.cuda.current_stream().cuda_stream
    if "handle" in st:
        x = st["x"]
        if case.get("op") == "trial":
            m.potential_eval_async(st["handle"], st["prec"], x.data_ptr(), x.numel(), e_dev_ptr=st["e"].data_ptr(),
                                   d_ptr=st["d"].data_ptr(), t=0.5, stream=stream)
            return dict(energy=st["e"])
        m.potential_eval_async(st["handle"], st["prec"], x.data_ptr(), x.numel(), g_ptr=st["g"].data_ptr(),
                               e_dev_ptr=st["e"].data_ptr(), stream=stream)
        return dict(energy=st["e"], gradient=st["g"])
    if kind == "batch":
        for s, x in zip(st["states"], st["x0"]):
            _set_coords(s, x)
        res = st["mini"].minimiseBatch(st["states"])
        return dict(coords=torch.cat([_coords(s) for s in st["states"]]),
                    energy=np.array([r["energy"] for r in res]))
    state, mini = st["state"], st["mini"]
    if case.get("host"):
        state.coords(st["x0"])
        return dict(coords=mini.minimise(state), energy=mini.stats["energy"])
    _set_coords(state, st["x0"])
    mini.minimise(state, download=False)
    out = dict(coords=_coords(state).clone())
    if kind == "relax":
        out["energy"] = mini.stats["energy"]
    return out


# ------------------------------------------------------------------- its work
def work(case):
    kind = case["kind"]
    b = 8 if case.get("prec", "fp64") == "fp64" else 4
    if kind in ("field", "elements", "pillars"):
        sites = case["nx"] * case["ny"] * case["nz"]
        n = sites * case.get("nf", 3)
        if case.get("op") == "trial":
            return dict(bytes=2 * n * b, flops=20 * n)  # x, d in
        return dict(bytes=2 * n * b + (sites if kind == "pillars" else 0), flops=30 * n)  # x in, g out (and the solid)
    if kind == "cluster":
        n, d = case["n"], case["dim"]
        return dict(bytes=2 * n * d * b, flops=n * (n - 1) / 2 * (10 + 5 * d))
    pairs = DENSITY * 4 / 3 * math.pi * RCUT ** 3 / 2  # per particle, each pair once
    if kind == "liquid":
        n = case["side"] ** 3
        return dict(bytes=6 * n * b, flops=25 * pairs * n)
    if kind == "sheet":
        nx, ny = case["nx"], case["ny"]
        bars = nx * (ny - 1) + ny * (nx - 1) + (nx - 1) * (ny - 1)
        hinges = bars - 2 * (nx - 1) - 2 * (ny - 1)
        # coordinates in, gradient out, the node ids of every bar and hinge
        return dict(bytes=6 * nx * ny * b + 8 * bars + 16 * hinges, flops=30 * bars + 200 * hinges)
    if kind == "fire":
        n = case["side"] ** 3
        # per step: x and v in and out, g out and in
        return dict(bytes=case["iters"] * 18 * n * b, flops=case["iters"] * (25 * pairs + 30) * n)
    if kind == "relax":
        n = case["nx"] * case["ny"] * case["nz"] * case["nf"]
        b = 4 if case["mode"] == "mixed" else 8
    else:
        n = sum(s * s for s in _batch_sides(case))
    # per iteration with P stored pairs: the direction and the Gram dots read
    # the pairs once each, g and d; the accepted step reads x and d and writes
    # x, g and y
    vec = sum(4 * min(k, 5) + 8 for k in range(case["iters"]))
    return dict(bytes=vec * n * b, flops=sum(16 * min(k, 5) + 60 for k in range(case["iters"])) * n)


def tolerance(case):
    """About four times the largest error against exact() over sizes, seeds
    and options of each kind (relative, and the largest entry's)."""
    kind, fp64 = case["kind"], case.get("prec", "fp64") == "fp64"
    if kind == "relax":  # rounding differences grow from iteration to iteration
        return dict(rel=1.5e-5, max=1.5e-4) if case["mode"] == "mixed" else dict(rel=1e-11, max=5e-10)
    if kind == "batch":
        return dict(rel=1e-9, max=2e-8)
    if kind == "fire":
        return dict(rel=2e-15, max=5e-14)
    if kind == "cluster":
        return dict(rel=1e-14, max=5e-14) if fp64 else dict(rel=3e-5, max=1.2e-4)
    if kind == "liquid":
        # FP32 positions in a box of up to 67 sigma: the difference of two
        # positions keeps few bits of a short pair's separation
        return dict(rel=3e-15, max=2e-14) if fp64 else dict(rel=3e-5, max=3e-3)
    if kind == "sheet":
        # FP64: the angle comes from an arc cosine, which loses half the digits
        # of a nearly flat hinge, as in the reference
        return dict(rel=1e-9, max=1e-6) if fp64 else dict(rel=1.6e-4, max=1e-3)
    return dict(rel=1e-15, max=5e-15) if fp64 else dict(rel=2.5e-7, max=1.5e-6)


# ------------------------------------------------------------------- in 64 bits
def _coefficients(nf, st, w):
    """kappa and kappaP of every fluid."""
    if nf <= 2:
        return [3 * st / w] * nf, [3 * st * w] * nf
    t = [st] * nf if np.isscalar(st) else st
    mix = ((1, 1, -1), (1, -1, 1), (-1, 1, 1))
    one = [0.5 * sum(s * v for s, v in zip(r, t)) for r in mix]
    return [6 * v / w for v in one], [6 * v * w for v in one]


class _Field:
    """Energy and projected gradient of a phase field by torch in FP64."""

    def __init__(self, shape, nf, st, w, solid=None, pressure=None, fixed=()):
        self.shape, self.nf, self.fixed, self.pressure = shape, nf, list(fixed), pressure
        self.kappa, self.kappaP = _coefficients(nf, st, w)
        self.vol, self.solid = 1.0, None
        if solid is not None:
            self.solid = solid
            self.vol = self._volumes(solid)

    @staticmethod
    def _volumes(s):
        """Node volumes beside solid nodes: eighths by the number of solid
        faces, edges and corners among the 26 neighbours."""
        faces, edges, corners = (torch.zeros(s.shape, dtype=torch.int32, device=s.device) for _ in range(3))
        axis = [torch.zeros_like(s) for _ in range(3)]
        across = [torch.zeros_like(s) for _ in range(3)]
        for dx in (-1, 0, 1):
            for dy in (-1, 0, 1):
                for dz in (-1, 0, 1):
                    o = (dx, dy, dz)
                    k = sum(v != 0 for v in o)
                    if k == 0:
                        continue
                    nb = torch.roll(s, (-dx, -dy, -dz), (0, 1, 2))
                    if k == 1:
                        faces += nb
                        a = [i for i in range(3) if o[i]][0]
                        axis[a] |= nb
                    elif k == 2:
                        edges += nb
                        a = [i for i in range(3) if not o[i]][0]
                        across[a] |= nb
                    else:
                        corners += nb
        flat = (axis[0] & ~across[0]) | (axis[1] & ~across[1]) | (axis[2] & ~across[2])
        t = torch.where(faces == 1, torch.where(flat, 4, 5), torch.where(faces == 2, 6, 7))
        t0 = torch.where(edges == 0, 1, torch.where(edges == 1, 2, 3))
        t = torch.where(faces == 0, torch.where((edges == 0) & (corners == 0), 8, t0), t)
        return torch.where(s, 0, t).double() / 8

    def energy_sites(self, c):
        """The energy of the field (a scalar with a graph when c has one)."""
        total = 0
        for k in range(self.nf):
            ck = c[..., k]
            if self.nf == 1:
                e = self.kappa[0] / 16 * self.vol * (ck + 1) ** 2 * (ck - 1) ** 2
                f = 0.25 * self.kappaP[0]
            else:
                e = 0.5 * self.kappa[k] * self.vol * ck ** 2 * (ck - 1) ** 2
                f = 0.5 * self.kappaP[k]
            g2 = 0
            for d in range(3):
                if self.shape[d] == 1:
                    continue
                dm, dp = ck - torch.roll(ck, 1, d), ck - torch.roll(ck, -1, d)
                if self.solid is None:
                    g2 = g2 + 0.5 * (dm ** 2 + dp ** 2)
                else:
                    sm, sp = torch.roll(self.solid, 1, d), torch.roll(self.solid, -1, d)
                    hm = torch.where(sm, 0.0, torch.where(sp, 1.0, 0.5))
                    hp = torch.where(sp, 0.0, torch.where(sm, 1.0, 0.5))
                    g2 = g2 + hm * dm ** 2 + hp * dp ** 2
            e = e + f * self.vol * g2
            if self.pressure and self.pressure[k]:
                e = e - self.pressure[k] * ck * self.vol
            total = total + e.sum()
        return total

    def energy(self, x):
        return float(self.energy_sites(x.reshape(*self.shape, self.nf)))

    def project(self, v):
        if self.nf > 1:
            v = v.reshape(-1, self.nf).clone()
            var = [k for k in range(self.nf) if k not in self.fixed]
            v[:, self.fixed] = 0
            v[:, var] -= v[:, var].sum(1, keepdim=True) / len(var)
        return v.reshape(-1)

    def eg(self, x):
        c = x.detach().reshape(*self.shape, self.nf).clone().requires_grad_(True)
        e = self.energy_sites(c)
        (g,) = torch.autograd.grad(e, c)
        return float(e.detach()), self.project(g.reshape(-1))


def _case_field(case):
    nf = case.get("nf", 3)
    kw = {}
    if case["kind"] == "pillars":
        kw = dict(solid=_pillar_solid(case), pressure=[0.0, 0.05, 0.0], fixed=[0])
    return _Field((case["nx"], case["ny"], case["nz"]), nf, SIGMA if nf == 3 else 1.0, 1.0 if nf == 1 else 2.0, **kw)


def _liquid_eg(x, side):
    """Truncated and shifted pairs by shifts of the lattice on which the
    particles started: a pair within the cutoff is at most three lattice
    steps apart along each axis."""
    L = side * LATTICE
    p = x.reshape(side, side, side, 3)
    g = torch.zeros_like(p)
    e = torch.zeros((), dtype=torch.float64, device=x.device)
    shift = 4 * (RCUT ** -12 - RCUT ** -6)
    for a in range(-3, 4):
        for b in range(-3, 4):
            for c in range(-3, 4):
                if (a, b, c) == (0, 0, 0):
                    continue
                dx = p - torch.roll(p, (a, b, c), (0, 1, 2))
                dx = dx - L * torch.round(dx / L)
                r2 = (dx * dx).sum(-1)
                near = r2 < RCUT ** 2
                i6 = torch.where(near, r2, 1.0) ** -3
                e += 0.5 * torch.where(near, 4 * (i6 * i6 - i6) - shift, 0.0).sum()
                g += dx * torch.where(near, -24 * (2 * i6 * i6 - i6) / torch.where(near, r2, 1.0), 0.0)[..., None]
    return float(e), g.reshape(-1)


def _cluster_eg(x, dim):
    p = x.reshape(-1, dim)
    dx = p[:, None, :] - p[None, :, :]
    r2 = (dx * dx).sum(-1)
    r2.fill_diagonal_(1.0)
    i6 = r2 ** -3
    pair, f = 4 * (i6 * i6 - i6), -24 * (2 * i6 * i6 - i6) / r2
    pair.fill_diagonal_(0.0)
    f.fill_diagonal_(0.0)
    return float(0.5 * pair.sum()), (dx * f[..., None]).sum(1).reshape(-1)


def _sheet_eg(x, nx, ny):
    """Bars of rest length one and hinges of rest angle pi; the stretching
    gradient is twice the derivative of its energy, as in the reference.
    Elements whose nodes are all clamped do not exist."""
    p = x.detach().reshape(nx, ny, 3).clone().requires_grad_(True)

    def length(u, v):
        return (u - v).norm(dim=-1) - 1.0

    bars = [length(p[1:, :], p[:-1, :]), length(p[1:, 1:], p[:-1, :-1]), length(p[1:-1, 1:], p[1:-1, :-1])]
    stretch = sum(0.5 * (b * b).sum() for b in bars)

    def hinge(x1, x2, x3, x4):
        # edge x2-x3 with the tips x1 and x4; the angle's deviation from flat
        b1, b2, b3 = x2 - x1, x3 - x2, x4 - x3
        n1, n2 = torch.linalg.cross(b1, b2), torch.linalg.cross(b2, b3)
        # theta - pi with the angle in (0, 2 pi): the atan2 of the opposite vector
        t = torch.atan2(-b2.norm(dim=-1) * (n1 * b3).sum(-1), -(n1 * n2).sum(-1))
        return 0.5 * 0.01 * (t * t).sum()

    a, b, c, d = p[:-1, :-1], p[1:, :-1], p[1:, 1:], p[:-1, 1:]
    bend = hinge(b, c, a, d)  # the diagonal of each square
    # vertical edges (i fixed) between square (i-1, j)'s lower triangle and (i, j)'s upper one
    bend = bend + hinge(p[:-2, :-1], p[1:-1, :-1], p[1:-1, 1:], p[2:, 1:])
    # horizontal edges (j fixed) between square (i, j-1)'s upper triangle and (i, j)'s lower one
    bend = bend + hinge(p[:-1, :-2], p[1:, 1:-1], p[:-1, 1:-1], p[1:, 2:])
    (gs,) = torch.autograd.grad(stretch, p)
    (gb,) = torch.autograd.grad(bend, p)
    g = 2 * gs + gb
    g[0] = 0
    g[-1] = 0
    return float((stretch + bend).detach()), g.reshape(-1)


def _lbfgs(f, x, iters, m_hist=5):
    """L-BFGS with the two-loop recursion and a backtracking line search."""
    e, g = f.eg(x)
    hist = []
    for _ in range(iters):
        if not hist:
            d = -g / g.norm()
        else:
            q, al = -g, []
            for s, y, rho in reversed(hist):
                al.append(rho * s.dot(q))
                q = q - al[-1] * y
            s, y, rho = hist[-1]
            q = q / (rho * y.dot(y))
            for (s, y, rho), a in zip(hist, reversed(al)):
                q = q + (a - rho * y.dot(q)) * s
            d = q
        d = f.project(d)
        gs = float(g.dot(d))
        tau = 1.0
        if gs > 0:
            gs, tau = -gs, -1.0
        t = -0.5 * gs
        for _ in range(10):
            if e - f.energy(x + tau * d) >= t:
                break
            tau, t = 0.5 * tau, 0.5 * t
        s = tau * d
        x = x + s
        gold = g
        e, g = f.eg(x)
        y = g - gold
        sy = s.dot(y)
        if float(sy) != 0:
            hist = (hist + [(s, y, 1 / sy)])[-m_hist:]
    return x, e


def _fire(side, x, iters, dt0=0.002, dt_max=0.02):
    _, g = _liquid_eg(x, side)
    v, a, dt, n = torch.zeros_like(x), 0.1, dt0, 0
    for _ in range(iters):
        p = -float(v.dot(g))
        if p > 0:
            v = (1 - a) * v - (a * v.norm() / g.norm() + dt) * g
            n += 1
            if n > 5:
                a, dt = a * 0.99, min(dt * 1.1, dt_max)
        else:
            v, n, a, dt = -dt * g, 0, 0.1, dt * 0.5
        x = x + dt * v
        _, g = _liquid_eg(x, side)
    return x


def exact(case, seed):
    kind, gen = case["kind"], _gen(seed)
    dtype = _DT[case.get("prec", "fp64")]
    if kind in ("field", "pillars", "elements"):
        x = (_pillar_input if kind == "pillars" else _field_input)(case, gen, dtype)
        f = _case_field(case)
        if case.get("op") == "trial":
            d = _uniform(gen, x.shape, -0.05, 0.05, dtype)
            return dict(energy=np.array([f.energy(x.double() + 0.5 * d.double())]))
        e, g = f.eg(x.double().reshape(-1))
        return dict(energy=np.array([e]), gradient=g.reshape(x.shape))
    if kind == "cluster":
        x = _cluster_input(case, gen, dtype)
        e, g = _cluster_eg(x.double(), case["dim"])
    elif kind == "liquid":
        x = _liquid_input(case, gen, dtype)
        e, g = _liquid_eg(x.double(), case["side"])
    elif kind == "sheet":
        x = _sheet_input(case, gen, dtype)
        e, g = _sheet_eg(x.double(), case["nx"], case["ny"])
    elif kind == "relax":
        x, e = _lbfgs(_case_field(case), _field_input(case, gen, torch.float32).double().reshape(-1), case["iters"])
        return dict(coords=x, energy=e)
    elif kind == "fire":
        x = _fire(case["side"], _liquid_input(case, gen, torch.float32).double().reshape(-1), case["iters"])
        return dict(coords=x)
    else:
        sides, widths, xs = _batch_instances(case, gen)
        got = [_lbfgs(_Field((s, s, 1), 1, 1.0, w), x, case["iters"]) for s, w, x in zip(sides, widths, xs)]
        return dict(coords=torch.cat([x for x, _ in got]), energy=np.array([e for _, e in got]))
    return dict(energy=np.array([e]), gradient=g.reshape(x.shape))
