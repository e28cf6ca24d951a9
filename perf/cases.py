"""The work that users of this package have it do, as timed cases.

Every case is one of seven kinds:

  steps       a weakly compressible SPH run: a `Solver` on `Particles`, a few
              RK2 or Euler time steps from a given state, then the fluid's
              state.  Dam breaks in 2D and 3D and the elliptical drop, in
              single and in double precision (the default of the reference).
  density     re-bin and summation density of a point set in the unit cube.
  forces      every neighbour sum of the scheme as a calc of its own (density,
              equation of state, density rate, momentum, XSPH), on a periodic
              box or with variable smoothing lengths: what integrators other
              than the fused ones and analysis scripts call.
  neighbours  the neighbour sets of every particle as a CSR.
  batch       many small scenes of uneven size advanced together.
  rollout     the edge-MLP surrogate advancing a 2D dam break, its check
              against the plain solver included.
  train       loss, backward pass and gradients of the surrogate on a graph.

Runs restart from the state that `prepare` made, so a pass can be repeated.
Results are returned in the particles' own (user) order.
"""
import math
import os

import numpy as np
import torch

import pysph_amd
import pysph_amd.base.api as base
import pysph_amd.solver.api as solver
import pysph_amd.sph.api as sph
from pysph_amd.batch.engine import BatchedWCSPH, scene_from_arrays
from pysph_amd.solver import generators as gen
from pysph_amd.surrogate.graph import ParticleGraph, combined_array
from pysph_amd.surrogate.model import EdgeMLP
from pysph_amd.surrogate.solver import SurrogateWCSPH, get_user, set_user

Fluid = base.ParticleType.Fluid
WEIGHTS = os.path.join(os.path.dirname(pysph_amd.__file__), "surrogate", "weights",
                       "dam2d_edge_mlp.npz")


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest runs: a step is some 20 launches on a few blocks each,
        # so latency counts.  A tutorial-sized 2D dam break in single precision
        dict(name="dam2d_f32_1k5", kind="steps", scene="dam2d", n=1500, precision="single",
             integrator="rk2", steps=20),
        # the reference's elliptical drop (5025 particles) in its default
        # double precision
        dict(name="drop_f64_5k", kind="steps", scene="drop", n=5025, precision="double",
             integrator="rk2", steps=20),
        # a 3D dam break of ordinary size in double precision
        dict(name="dam3d_f64_60k", kind="steps", scene="dam3d", n=60000, precision="double",
             integrator="rk2", steps=3),
        # the benchmark: 1.06M fluid and 0.35M boundary particles, single
        dict(name="dam3d_f32_1m", kind="steps", scene="dam3d", n=1062882, precision="single",
             integrator="rk2", steps=3),
        # neighbour search and density of a large random set, single precision
        dict(name="cube_f32_4m", kind="density", points="uniform", n=4194301,
             precision="single"),
        # the same of a clustered set in double precision (uneven cells)
        dict(name="cube_f64_clustered_300k", kind="density", points="clustered", n=300007,
             precision="double"),
        # the scheme's sums one by one in a fully periodic 3D box
        dict(name="forces_f32_periodic_100k", kind="forces", dim=3, n=100000,
             precision="single", periodic=True, varh=False),
        # the same with smoothing lengths that vary by a factor of two
        dict(name="forces_f64_varh_40k", kind="forces", dim=2, n=40000, precision="double",
             periodic=False, varh=True),
        # neighbour lists of every particle, as the locators hand them out
        dict(name="neighbours_f64_50k", kind="neighbours", dim=3, n=50021, precision="double",
             varh=False),
        # 48 scenes of 1k to 64k particles per launch
        dict(name="batch_48", kind="batch", n=48, steps=4),
        # a surrogate run of ten steps (the tenth is checked)
        dict(name="rollout_40k", kind="rollout", n=40000, steps=10),
        # one training step on one graph
        dict(name="train_30k", kind="train", n=30000),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["steps", "steps", "steps", "density", "forces", "neighbours", "batch",
                       "rollout", "train"])
    prec = rng.choice(["single", "double"])
    if kind == "steps":
        scene = rng.choice(["dam2d", "drop", "dam3d"])
        integ = rng.choice(["rk2", "rk2", "rk2", "euler"])
        if scene == "dam3d":
            n = _log(rng, 5000, 1000000 if prec == "single" else 100000)
            return dict(kind=kind, scene=scene, n=n, precision=prec, integrator=integ, steps=3)
        n = _log(rng, 800, 100000)
        return dict(kind=kind, scene=scene, n=n, precision=prec, integrator=integ, steps=20)
    if kind == "density":
        n = _log(rng, 10000, 4000000 if prec == "single" else 400000)
        return dict(kind=kind, points=rng.choice(["uniform", "clustered"]), n=n, precision=prec)
    if kind == "forces":
        how = rng.choice(["periodic", "varh", "plain"])
        return dict(kind=kind, dim=rng.choice([2, 3]), n=_log(rng, 4000, 200000),
                    precision=prec, periodic=how == "periodic", varh=how == "varh")
    if kind == "neighbours":
        return dict(kind=kind, dim=rng.choice([2, 3]), n=_log(rng, 3000, 60000),
                    precision=prec, varh=rng.random() < 0.3)
    if kind == "batch":
        return dict(kind=kind, n=_log(rng, 6, 48), steps=4)
    if kind == "rollout":
        return dict(kind=kind, n=_log(rng, 20000, 60000), steps=10)
    return dict(kind=kind, n=_log(rng, 20000, 60000))


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _rng(seed):
    return np.random.Generator(np.random.PCG64(int(seed)))


def _scene(case, seed):
    """(fluid, boundary or None, info): the generators' lattices with
    positions jittered by a few per cent of the spacing."""
    rng = _rng(seed)
    n, prec = case["n"], case["precision"]
    if case["scene"] == "drop":
        f, b, info = gen.elliptical_drop_2d(n, aspect=0.9, precision=prec)
        m = f.get_number_of_particles()
        f.set(x=f.get("x") + 0.02 * info["dx"] * rng.uniform(-1, 1, m),
              y=f.get("y") + 0.02 * info["dx"] * rng.uniform(-1, 1, m))
        return f, b, info
    if case["scene"] == "dam2d":
        return gen.dam_break_2d(width=0.5, height=1.0, dx=math.sqrt(0.5 / n), jitter=0.02,
                                seed=int(seed), precision=prec)
    s = (n / 1062882.0) ** (1.0 / 3.0)
    col = tuple(max(4, int(round(k * s))) for k in (81, 81, 162))
    tank = (max(col[0] + 2, int(round(216 * s))), col[1], col[2])
    return gen.dam_break_3d(dx=1.0 / (135 * s), column=col, tank=tank, jitter=0.02,
                            seed=int(seed), precision=prec)


def _box(case, seed, view=None):
    """A jittered lattice of about n particles in a box with random
    velocities, and its box lengths."""
    rng = _rng(seed)
    dim, n = case["dim"], case["n"]
    k = n ** (1.0 / dim)
    nx, ny = int(round(1.2 * k)), int(round(k))
    nz = 1 if dim == 2 else max(6, int(round(n / (nx * ny))))
    ny = ny if dim == 3 else max(6, int(round(n / nx)))
    dx = 1.0 / nx
    i, j, l = np.meshgrid(np.arange(nx), np.arange(ny), np.arange(nz), indexing="ij")
    pos = [(a.ravel() + 0.5) * dx + 0.15 * dx * rng.uniform(-1, 1, i.size) for a in (i, j, l)]
    if dim == 2:
        pos[2] = np.zeros(i.size)
    m = i.size
    vel = [rng.normal(0.0, 1.0, m) for _ in range(dim)] + [np.zeros(m)] * (3 - dim)
    h = 1.2 * dx * ((1.0 + rng.random(m)) if case.get("varh") else np.ones(m))
    if view is not None:
        # the same set, mirrored and numbered from another particle on
        r = _rng(view)
        pos = [p * float(r.choice([-1.0, 1.0])) for p in pos]
        k = int(r.integers(m))
        pos, h = [np.roll(p, k) for p in pos], np.roll(h, k)
    pa = base.get_particle_array(
        cl_precision=case["precision"], name="fluid", type=Fluid, x=pos[0], y=pos[1], z=pos[2],
        u=vel[0], v=vel[1], w=vel[2], h=h, m=np.full(m, 1000.0 * dx ** dim),
        rho=np.full(m, 1000.0))
    return pa, (nx * dx, ny * dx, nz * dx)


def _batch_scenes(case, seed):
    """Drops and dam breaks of the batched benchmark, jittered."""
    rng = _rng(seed)
    scenes = gen.batch_scenes(n_scenes=case["n"], seed=case["n"])
    for f, _, info in scenes:
        m = f.get_number_of_particles()
        f.set(x=f.get("x") + 0.02 * info["dx"] * rng.uniform(-1, 1, m),
              y=f.get("y") + 0.02 * info["dx"] * rng.uniform(-1, 1, m))
    return scenes


def _dam(case, seed):
    """A 2D dam break with boundary as the surrogate is trained on (widths
    0.3 to 1 m, heights 0.5 to 2 m), in motion."""
    rng = _rng(seed)
    width, height = 0.6, 1.0
    f, b, info = gen.dam_break_2d(width=width, height=height,
                                  dx=math.sqrt(width * height / case["n"]), jitter=0.02,
                                  seed=int(seed))
    m = f.get_number_of_particles()
    x, y = f.get("x") / width, f.get("y") / height
    s = 0.3 * math.sqrt(2.0 * 9.81 * height)
    f.set(u=s * x * (1.0 - y) + 0.002 * s * rng.normal(size=m),
          v=-s * y * (1.0 - x) + 0.002 * s * rng.normal(size=m))
    return f, b, info


STATE3 = ("x", "y", "z", "u", "v", "w")


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case}
    if kind == "steps":
        f, b, info = _scene(case, seed)
        dim = 3 if case["scene"] == "dam3d" else 2
        st["f"], st["b"], st["info"] = f, b, info
        names = [STATE3[k] for k in range(6) if k % 3 < dim]
        st["init"] = {k: f.get_carray(k).clone() for k in names}
        particles = base.Particles([f] + ([b] if b is not None else []))
        s = solver.wcsph_solver(dim, integrator=case["integrator"], co=info["co"],
                                ro=info["rho0"], gamma=info["gamma"], alpha=info["alpha"],
                                beta=info["beta"], eta=info["eta"], gravity=info["g"],
                                xsph_eps=info["eps"] or None, with_solid=b is not None)
        s.setup_integrator(particles)
        s.set_time_step(info["dt"])
        s.set_print_freq(0)
        st["solver"] = s
    elif kind == "density":
        pa = gen.cube_array(case["n"], kind=case["points"], seed=int(seed),
                            precision=case["precision"])
        st["pa"] = pa
        particles = base.Particles([pa])
        op = solver.SPHOperation(sph.SPHRho.withargs(), on_types=[Fluid], from_types=[Fluid],
                                 updates=["rho"], id="density")
        st["calc"] = op.get_calcs(particles, base.CubicSplineKernel(dim=3))[0]
    elif kind == "forces":
        pa, box = _box(case, seed)
        dim = case["dim"]
        st["pa"] = pa
        dom = None
        if case["periodic"]:
            dom = base.PeriodicDomain(xmin=0.0, xmax=box[0], ymin=0.0, ymax=box[1],
                                      **(dict(zmin=0.0, zmax=box[2]) if dim == 3 else {}))
        particles = base.Particles([pa], variable_h=case["varh"], periodic_domain=dom)
        for nm in ("arho", "ax", "ay", "az", "dx", "dy", "dz"):
            pa.add_property({"name": nm})
        ker = base.CubicSplineKernel(dim=dim)
        vel, pos = ["u", "v", "w"][:dim], ["x", "y", "z"][:dim]
        F = [Fluid]
        st["ops"] = [(op.get_calcs(particles, ker)[0], out) for op, out in (
            (solver.SPHOperation(sph.SPHRho.withargs(), on_types=F, from_types=F,
                                 updates=["rho"], id="rho"), ["rho"]),
            (solver.SPHOperation(sph.TaitEquation.withargs(co=30.0, ro=1000.0, gamma=7.0),
                                 on_types=F, updates=["p", "cs"], id="eos"), ["p", "cs"]),
            (solver.SPHIntegration(sph.SPHDensityRate.withargs(hks=False), on_types=F,
                                   from_types=F, updates=["rho"], id="rate"), ["arho"]),
            (solver.SPHIntegration(sph.MomentumEquation.withargs(alpha=0.5, beta=0.5, eta=0.1,
                                                                 dim=dim),
                                   on_types=F, from_types=F, updates=vel, id="mom"),
             ["ax", "ay", "az"][:dim]),
            (solver.SPHIntegration(sph.XSPHCorrection.withargs(eps=0.5, dim=dim), on_types=F,
                                   from_types=F, updates=pos, id="xsph"),
             ["dx", "dy", "dz"][:dim]))]
        st["outs"] = ["rho", "p", "cs", "arho"] + st["ops"][3][1] + st["ops"][4][1]
    elif kind == "neighbours":
        # one set per size, so that every seed has as many neighbours
        pa, _ = _box(case, case["n"], view=seed)
        st["pa"] = pa
        particles = base.Particles([pa], variable_h=case["varh"])
        st["loc"] = particles.nnps_manager.get_neighbor_particle_locator(pa, pa, 2.0)
    elif kind == "batch":
        scenes = [scene_from_arrays(f, b, info) for f, b, info in _batch_scenes(case, seed)]
        with torch.cuda.stream(_side_stream()):
            eng = BatchedWCSPH(scenes)
            st["init"] = {k: t.clone() for k, t in eng.fa.items()}
            off = np.repeat(eng.f_off[:-1], np.diff(eng.f_off))
            st["off"] = torch.from_numpy(off).to(eng.fa["uid"].device)
            eng.step()
            eng.capture()
        st["engine"] = eng
    elif kind == "rollout":
        f, b, info = _dam(case, seed)
        st["sur"] = SurrogateWCSPH(f, b, info, EdgeMLP.load(WEIGHTS))
        st["init"] = st["sur"].state()
    elif kind == "train":
        f, b, info = _dam(case, seed)
        rng = _rng(seed + 1)
        g = ParticleGraph(combined_array(f, b), info, domain=info["domain"])
        st["graph"], st["model"] = g, EdgeMLP.load(WEIGHTS)
        st["init"] = {k: g.pa.get_carray(k).clone() for k in ("x", "y", "u", "v")}
        tgt = torch.from_numpy(_target(g.n, g.n_fluid, rng)).to(g.device)
        st["target"] = tgt
        st["out"] = torch.empty((g.n, 2), dtype=torch.float32, device=g.device)
    else:
        raise ValueError(kind)
    return st


def _target(n, nf, rng):
    t = np.zeros((n, 2), dtype=np.float32)
    t[:nf] = rng.normal(0.0, 0.5, (nf, 2)) + np.array([0.0, -1.0])
    return t


_stream = None


def _side_stream():
    """The stream a program that replays the batch's graph runs on."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "steps":
        f, b, s = st["f"], st["b"], st["solver"]
        for k, t in st["init"].items():
            set_user(f, k, t)
        s.t = 0.0
        s.set_final_time(s.dt * (case["steps"] - 0.5))
        s.solve()
        out = {k: get_user(f, k) for k in list(st["init"]) + ["rho", "p"]}
        if b is not None:
            out["rho_b"] = get_user(b, "rho")
        return out
    if kind == "density":
        st["pa"].set_dirty(True)
        st["calc"].sph("rho")
        return {"rho": get_user(st["pa"], "rho")}
    if kind == "forces":
        st["pa"].set_dirty(True)
        for calc, outs in st["ops"]:
            calc.sph(*outs)
        return {k: get_user(st["pa"], k) for k in st["outs"]}
    if kind == "neighbours":
        st["pa"].set_dirty(True)
        off, nbr = st["loc"].get_csr()
        return {"off": off, "nbr": nbr}
    if kind == "batch":
        eng = st["engine"]
        with torch.cuda.stream(_side_stream()):
            for k, t in st["init"].items():
                eng.fa[k].copy_(t)
            eng.run(case["steps"])
            idx = st["off"] + eng.fa["uid"][:eng.nf].long()
            out = {}
            for k in ("x", "y", "u", "v", "rho", "p"):
                out[k] = torch.empty(eng.nf, dtype=torch.float32, device=eng.device)
                out[k][idx] = eng.fa[k][:eng.nf]
        return out
    if kind == "rollout":
        sur = st["sur"]
        sur.reset(st["init"])
        sur.run(case["steps"])
        return sur.state()
    g, model = st["graph"], st["model"]
    g.set_state(st["init"])
    g.build()
    model.zero_grad(torch.cuda.current_stream().cuda_stream)
    loss = model.loss_backward(g, g.user_rows_to_slot(st["target"]), out=st["out"])
    return {"loss": loss, "out": g.slot_rows_to_user(st["out"]), "grads": model.grads()}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _nbrs(hdx, dim):
    """Neighbours within 2h at rest density."""
    r = 2.0 * hdx
    return math.pi * r * r if dim == 2 else 4.0 / 3.0 * math.pi * r ** 3


def work(case):
    """Bytes: each particle property that a step (or sum) has to read or
    write, once.  Flops: 20 a density pair, 80 a momentum + XSPH pair."""
    kind = case["kind"]
    sz = 8 if case.get("precision") == "double" else 4
    n = case["n"]
    if kind == "steps":
        dim = 3 if case["scene"] == "dam3d" else 2
        nb = {"drop": 0.0, "dam2d": 3 * 3 * 4.0 * math.sqrt(2.0 * n),
              "dam3d": 352458 * (n / 1062882.0) ** (2.0 / 3.0)}[case["scene"]]
        per = {3: (264 / 4, 120 / 4), 2: (208 / 4, 112 / 4)}[dim]
        stages = 2 if case["integrator"] == "rk2" else 1
        nn = _nbrs(1.2 if dim == 3 else 1.3, dim)
        one = sz * (per[0] * n + per[1] * nb) * stages / 2
        flops = stages * nn * (20.0 * (n + nb) + 80.0 * n)
        return {"bytes": case["steps"] * one, "flops": case["steps"] * flops}
    if kind == "density":
        return {"bytes": 10.0 * sz * n, "flops": 20.0 * 50 * n}
    if kind == "forces":
        nn = _nbrs(1.8 if case["varh"] else 1.2, case["dim"])
        return {"bytes": 40.0 * sz * n, "flops": 140.0 * nn * n}
    if kind == "neighbours":
        nn = _nbrs(1.8 if case["varh"] else 1.2, case["dim"])
        return {"bytes": n * (4.0 * sz + 8.0 + 8.0 * nn), "flops": 8.0 * nn * n}
    if kind == "batch":
        m = n * 15200.0  # mean of the log-uniform scene sizes
        return {"bytes": case["steps"] * 208.0 * m,
                "flops": case["steps"] * 2 * 100.0 * _nbrs(1.35, 2) * m}
    edges = 21.0 * n
    fwd = n * 2.0 * (16 * 128 + 2 * (128 * 256 + 256 * 128) + 256) + edges * 2 * 2 * 16 * 128
    if kind == "rollout":
        return {"bytes": case["steps"] * 64.0 * n, "flops": case["steps"] * fwd}
    return {"bytes": 64.0 * n + 8.0 * 138116, "flops": 3.0 * fwd}


def tolerance(case):
    """About four times the difference between a pass and the same sums in
    64 bits (for 64-bit storage: in another order), see `exact`."""
    kind = case["kind"]
    double = case.get("precision") == "double"
    if kind == "neighbours":
        return "exact"
    if kind == "steps":
        return {"rel": 2.5e-12, "max": 2e-11} if double else {"rel": 8e-4, "max": 1.2e-2}
    if kind == "density":
        return {"rel": 2.5e-15, "max": 1.5e-14} if double else {"rel": 6e-7, "max": 4e-6}
    if kind == "forces":
        return {"rel": 3.2e-14, "max": 1.5e-13} if double else {"rel": 1.4e-5, "max": 7e-5}
    if kind == "batch":
        return {"rel": 8e-4, "max": 1.2e-2}
    if kind == "rollout":
        # against the FP32 edge aggregation
        return {"rel": 7e-3, "max": 3.5e-1}
    return {"rel": 1.5e-2, "max": 6e-1}


# ---------------------------------------------------------------------------
# the same in 64 bits, plain torch
# ---------------------------------------------------------------------------
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _f64(pa, names):
    """Stored values of a particle array in user order, as float64."""
    return {k: torch.from_numpy(np.ascontiguousarray(pa.get(k, only_real_particles=False)))
            .to(_dev()).double() for k in names}


class _Cells:
    """Points sorted by cells of at least `radius`; pairs(dst, ...) yields
    (i, j, r_i - r_j, d2) of every pair closer than the pair's radius."""

    def __init__(self, pos, radius, period=None):
        self.pos, self.radius, self.period = pos, float(radius), period
        dev = pos.device
        lo, hi = pos.amin(0), pos.amax(0)
        size, dims, base_ = [], [], []
        for a in range(3):
            L = period[a] if period else 0.0
            if L:
                k = max(1, int(L / radius))
                size.append(L / k)
                dims.append(k)
                base_.append(0.0)
            else:
                size.append(float(radius))
                dims.append(int((float(hi[a]) - float(lo[a])) / radius) + 1)
                base_.append(float(lo[a]))
        self.size = torch.tensor(size, device=dev, dtype=torch.float64)
        self.lo = torch.tensor(base_, device=dev, dtype=torch.float64)
        self.dims = dims
        key = self._key(self._cell(pos, clamp=True))
        key, self.order = torch.sort(key, stable=True)
        n = dims[0] * dims[1] * dims[2]
        self.start = torch.searchsorted(key, torch.arange(n + 1, device=dev))

    def _cell(self, p, clamp=False):
        c = torch.floor((p - self.lo) / self.size).long()
        if clamp:
            for a in range(3):
                c[:, a].clamp_(0, self.dims[a] - 1)
        return c

    def _key(self, c):
        return (c[:, 2] * self.dims[1] + c[:, 1]) * self.dims[0] + c[:, 0]

    def pairs(self, dst, r2_of, chunk=150000):
        """r2_of(i, j): squared radius of each candidate pair."""
        three = self.dims[2] > 1 or (self.period and self.period[2])
        off = [(a, b, c) for c in ((-1, 0, 1) if three else (0,)) for b in (-1, 0, 1)
               for a in (-1, 0, 1)]
        for i0 in range(0, len(dst), chunk):
            p = dst[i0:i0 + chunk]
            cell = self._cell(p)
            ids = torch.arange(i0, i0 + len(p), device=p.device)
            for o in off:
                c = cell + torch.tensor(o, device=p.device)
                ok = torch.ones(len(p), dtype=torch.bool, device=p.device)
                for a in range(3):
                    if self.period and self.period[a]:
                        c[:, a] %= self.dims[a]
                    else:
                        ok &= (c[:, a] >= 0) & (c[:, a] < self.dims[a])
                k = torch.where(ok, self._key(c), torch.zeros_like(ids))
                s = self.start[k]
                cnt = torch.where(ok, self.start[k + 1] - s, torch.zeros_like(s))
                tot = int(cnt.sum())
                if not tot:
                    continue
                i = torch.repeat_interleave(ids, cnt, output_size=tot)
                first = torch.cumsum(cnt, 0) - cnt
                j = torch.arange(tot, device=p.device) + torch.repeat_interleave(
                    s - first, cnt, output_size=tot)
                j = self.order[j]
                d = dst[i] - self.pos[j]
                for a in range(3):
                    L = self.period[a] if self.period else 0.0
                    if L:
                        d[:, a] -= L * torch.round(d[:, a] / L)
                d2 = (d * d).sum(1)
                keep = torch.nonzero(d2 < r2_of(i, j)).flatten()
                yield i[keep], j[keep], d[keep], d2[keep]


def _w(q, h, dim):
    fac = 10.0 / (7.0 * math.pi) / h ** 2 if dim == 2 else 1.0 / math.pi / h ** 3
    t = (2.0 - q).clamp_min(0.0)
    return fac * torch.where(q > 1.0, 0.25 * t ** 3, 1.0 - 1.5 * q * q * (1.0 - 0.5 * q))


def _gw(q, r, h, dim):
    """grad W = r_ab * this."""
    fac = 10.0 / (7.0 * math.pi) / h ** 2 if dim == 2 else 1.0 / math.pi / h ** 3
    t = (2.0 - q).clamp_min(0.0)
    outer = -0.75 * t * t / (h * r.clamp_min(1e-300))
    inner = torch.where(q > 1e-14, 3.0 * (0.75 * q - 1.0) / (h * h), torch.zeros_like(q))
    return fac * torch.where(q >= 1.0, outer, inner)


def _pos(d):
    return torch.stack([d["x"], d["y"], d["z"]], 1)


def _vel(d):
    return torch.stack([d["u"], d["v"], d["w"]], 1)


def _sweep(dsts, srcs, body, sym=False, period=None, cells=None):
    """body(k, i, s, j, d, d2, h_ab) for every pair of destination set k and
    source set s."""
    rmax = 2.0 * max(float(a["h"].max()) for a in dsts + srcs) * (1.0 + 1e-12)
    for s, S in enumerate(srcs):
        C = _Cells(_pos(S), rmax, period)
        for k, D in enumerate(dsts):
            def r2(i, j):
                hd = D["h"][i]
                return (2.0 * (torch.maximum(hd, S["h"][j]) if sym else hd)) ** 2
            for i, j, d, d2 in C.pairs(_pos(D), r2):
                body(k, i, s, j, d, d2, 0.5 * (D["h"][i] + S["h"][j]))


def _density(sets, dim, **kw):
    rho = [torch.zeros_like(a["h"]) for a in sets]

    def body(k, i, s, j, d, d2, h):
        rho[k].index_add_(0, i, sets[s]["m"][j] * _w(torch.sqrt(d2) / h, h, dim))
    _sweep(sets, sets, body, **kw)
    return rho


def _tait(rho, co, ro, gamma):
    r = rho / ro
    return co * co * ro / gamma * (r ** gamma - 1.0), co * r ** (0.5 * (gamma - 1.0))


def _momentum(D, srcs, dim, alpha, beta, eta, eps, **kw):
    """Accelerations from every source, XSPH (from the sources flagged) and
    the density rate of destination D."""
    n = len(D["h"])
    acc = torch.zeros((n, 3), dtype=torch.float64, device=D["h"].device)
    dv, rate = torch.zeros_like(acc), torch.zeros_like(D["h"])
    vd = _vel(D)
    vs = [_vel(S) for S in srcs]

    def body(k, i, s, j, d, d2, h):
        S = srcs[s]
        r = torch.sqrt(d2)
        g = _gw(r / h, r, h, dim)
        v = vd[i] - vs[s][j]
        dot = (v * d).sum(1)
        m, rho = S["m"][j], 0.5 * (D["rho"][i] + S["rho"][j])
        mu = h * dot / (d2 + eta * eta * h * h)
        visc = (-alpha * 0.5 * (D["cs"][i] + S["cs"][j]) * mu + beta * mu * mu) / rho
        tmp = D["p"][i] / D["rho"][i] ** 2 + S["p"][j] / S["rho"][j] ** 2
        tmp = tmp + torch.where(dot < 0.0, visc, torch.zeros_like(visc))
        acc.index_add_(0, i, (-m * tmp * g)[:, None] * d)
        rate.index_add_(0, i, m * dot * g)
        if S.get("xsph", True):
            dv.index_add_(0, i, (-eps * m * _w(r / h, h, dim) / rho)[:, None] * v)
    _sweep([D], srcs, body, **kw)
    return acc, dv, rate


FIELDS = ("x", "y", "z", "u", "v", "w", "h", "m")


def _advance(f, b, info, dim, integrator, steps):
    """RK2 (Heun) or Euler steps of the scheme; f, b: dicts of float64."""
    sets = [f] + ([b] if b is not None else [])
    for k, a in enumerate(sets):
        a["xsph"] = k == 0
    g = torch.tensor(info["g"] or (0.0, 0.0, 0.0), dtype=torch.float64, device=f["x"].device)
    dt = info["dt"]

    def rhs():
        for a, rho in zip(sets, _density(sets, dim)):
            a["rho"] = rho
            a["p"], a["cs"] = _tait(rho, info["co"], info["rho0"], info["gamma"])
        a, dv, _ = _momentum(f, sets, dim, info["alpha"], info["beta"], info["eta"],
                             info["eps"] or 0.0)
        return _vel(f) + dv, a + g

    def put(x, u):
        for k in range(dim):
            f["xyz"[k]], f["uvw"[k]] = x[:, k].contiguous(), u[:, k].contiguous()
    for _ in range(steps):
        x0, u0 = _pos(f), _vel(f)
        kx, ku = rhs()
        put(x0 + dt * kx, u0 + dt * ku)
        if integrator == "rk2":
            kx2, ku2 = rhs()
            put(x0 + 0.5 * dt * (kx + kx2), u0 + 0.5 * dt * (ku + ku2))


def exact(case, seed):
    kind = case["kind"]
    if kind == "steps":
        f, b, info = _scene(case, seed)
        dim = 3 if case["scene"] == "dam3d" else 2
        F = _f64(f, FIELDS)
        B = _f64(b, FIELDS) if b is not None else None
        _advance(F, B, info, dim, case["integrator"], case["steps"])
        out = {STATE3[k]: F[STATE3[k]] for k in range(6) if k % 3 < dim}
        out.update(rho=F["rho"], p=F["p"])
        if B is not None:
            out["rho_b"] = B["rho"]
        return out
    if kind == "density":
        pa = gen.cube_array(case["n"], kind=case["points"], seed=int(seed),
                            precision=case["precision"])
        return {"rho": _density([_f64(pa, FIELDS)], 3)[0]}
    if kind == "forces":
        pa, box = _box(case, seed)
        dim = case["dim"]
        D = _f64(pa, FIELDS)
        period = None
        if case["periodic"]:
            period = (box[0], box[1], box[2] if dim == 3 else 0.0)
            for k in range(dim):
                D["xyz"[k]] %= period[k]
        kw = dict(sym=case["varh"], period=period)
        D["rho"] = _density([D], dim, **kw)[0]
        D["p"], D["cs"] = _tait(D["rho"], 30.0, 1000.0, 7.0)
        a, dv, rate = _momentum(D, [D], dim, 0.5, 0.5, 0.1, 0.5, **kw)
        out = {"rho": D["rho"], "p": D["p"], "cs": D["cs"], "arho": rate}
        for k in range(dim):
            out["a" + "xyz"[k]], out["d" + "xyz"[k]] = a[:, k], dv[:, k]
        return out
    if kind == "batch":
        outs = []
        for f, b, info in _batch_scenes(case, seed):
            F = _f64(f, FIELDS)
            _advance(F, _f64(b, FIELDS) if b is not None else None, info, 2, "rk2",
                     case["steps"])
            outs.append(F)
        return {k: torch.cat([F[k] for F in outs]) for k in ("x", "y", "u", "v", "rho", "p")}
    if kind == "train":
        return _exact_train(case, seed)
    return None  # neighbours: whole numbers; rollout: rounding in 16 bits travels on


# ---- the network ----------------------------------------------------------
def _params(theta):
    shapes = [("w_in", 16, 128), ("b_in", 128)]
    for r in "01":
        shapes += [("w_ab" + r, 128, 256), ("w_c" + r, 16, 128), ("b_e" + r, 128),
                   ("w_u" + r, 256, 128), ("c_u" + r, 128)]
    shapes += [("w_out", 128, 2), ("b_out", 4)]
    out, o = {}, 0
    for name, *s in shapes:
        k = int(np.prod(s))
        out[name] = theta[o:o + k].reshape(s)
        o += k
    return out


def _exact_train(case, seed):
    f, b, info = _dam(case, seed)
    F, B = _f64(f, FIELDS), _f64(b, FIELDS)
    nf = len(F["x"])
    D = {k: torch.cat([F[k], B[k]]) for k in FIELDS}
    n = len(D["x"])
    rho = _density([D], 2)[0]
    co, ro, gam, alpha, eta = info["co"], info["rho0"], info["gamma"], info["alpha"], info["eta"]
    U, g, rs = co / 10.0, 9.81, 10.0
    got = []
    _sweep([D], [D], lambda k, i, s, j, d, d2, h: got.append((i, j, d, d2, h)))
    i, j, d, d2, h = (torch.cat([x[k] for x in got]) for k in range(5))
    r = torch.sqrt(d2)
    w, gf = _w(r / h, h, 2), _gw(r / h, r, h, 2)
    vel = _vel(D)
    dv = vel[i] - vel[j]
    p, cs = _tait(rho, co, ro, gam)
    m = 0.5 * (D["m"][i] + D["m"][j])
    pt = -m * (p[i] / rho[i] ** 2 + p[j] / rho[j] ** 2) * gf / g
    dot = (dv * d).sum(1)
    mu = h * dot / (d2 + eta * eta * h * h)
    visc = m * alpha * 0.5 * (cs[i] + cs[j]) * mu / (0.5 * (rho[i] + rho[j])) * gf / g
    visc = torch.where(dot < 0.0, visc, torch.zeros_like(visc))
    ps = 2.0 * g * h / U ** 2
    E = torch.zeros((len(i), 16), dtype=torch.float64, device=r.device)
    for k, v in enumerate((d[:, 0] / h, d[:, 1] / h, r / h, dv[:, 0] / U, dv[:, 1] / U,
                           (rho[i] / ro - 1.0) * rs, (rho[j] / ro - 1.0) * rs, w * h * h,
                           pt * d[:, 0] * ps, pt * d[:, 1] * ps, visc * d[:, 0] * ps,
                           visc * d[:, 1] * ps, torch.ones_like(r))):
        E[:, k] = v
    acc = torch.zeros((n, 4), dtype=torch.float64, device=r.device)
    acc.index_add_(0, i, torch.stack([pt * d[:, 0], pt * d[:, 1], visc * d[:, 0],
                                      visc * d[:, 1]], 1))
    X = torch.zeros((n, 16), dtype=torch.float64, device=r.device)
    X[:, 0], X[:, 1], X[:, 2] = D["u"] / U, D["v"] / U, (rho / ro - 1.0) * rs
    X[:, 3] = p * gam / (co * co * ro)
    X[nf:, 4] = 1.0
    X[:, 5] = 1.0
    X[:, 6:10] = 0.01 * acc
    with np.load(WEIGHTS, allow_pickle=False) as z:
        theta = torch.from_numpy(z["params"]).to(r.device).double().requires_grad_(True)
    P = _params(theta)
    H = torch.relu(X @ P["w_in"] + P["b_in"])
    for k in "01":
        PQ = H @ P["w_ab" + k]
        S = torch.relu(PQ[i, :128] + PQ[j, 128:] + E @ P["w_c" + k] + P["b_e" + k])
        A = torch.zeros((n, 128), dtype=torch.float64, device=r.device).index_add(0, i, S)
        H = H + torch.relu(torch.cat([H, A], 1) @ P["w_u" + k] + P["c_u" + k])
    Y = H @ P["w_out"] + P["b_out"][:2] + acc[:, :2] + acc[:, 2:]
    T = torch.from_numpy(_target(n, nf, _rng(seed + 1))).to(r.device).double()
    loss = ((Y[:nf] - T[:nf]) ** 2).sum() / nf
    loss.backward()
    return {"loss": loss.detach().reshape(1), "out": Y.detach(), "grads": theta.grad}
