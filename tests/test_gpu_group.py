"""The SoA passes' group scan (4, 8 or 16 lanes per destination) at the sizes
where it can go wrong, against the FP64 oracle on the same stored bits.

The lanes of a group share a list of stencil rows and a queue of accepted
sources in LDS, both flushed when nearly full: particle counts around whole
waves and around the sizes where the lane count changes, more rows than the
list holds (bins much smaller than the search radius), more neighbours than
the queue holds (dense points), one and two sources, far coordinates that the
FP32 cull cannot represent.  FP64 storage within 1e-12 (sums of at most 1e3
terms of one sign per particle: 1e3 * 2^-53 = 1.1e-13 relative; accelerations
normwise)."""
import numpy as np
import pytest
import torch

import pysph_amd.base.api as base
import pysph_amd.solver.api as solver
import pysph_amd.sph.api as sph
from oracle import oracle as O
from tests.util import max_rel, rel_norm, to_oracle

pytestmark = pytest.mark.gpu
Fluid = base.ParticleType.Fluid
Solid = base.ParticleType.Solid


def _points(n, dim, h, seed, ptype, spread=1.0, at=0.0):
    rng = np.random.Generator(np.random.PCG64(seed))
    pos = at + spread * rng.random((3, n))
    pos[dim:] = 0.0
    vel = rng.normal(size=(3, n))
    vel[dim:] = 0.0
    return base.get_particle_array(
        name="p%d" % seed, type=ptype, x=pos[0], y=pos[1], z=pos[2], u=vel[0], v=vel[1],
        w=vel[2], h=np.full(n, h), m=0.5 + rng.random(n), rho=1000.0 + 10 * rng.random(n),
        p=1e3 * rng.random(n), cs=10.0 + rng.random(n))


def _check(arrays, dim, min_cell_size=-1, varh=False):
    f = arrays[0]
    particles = base.Particles(arrays, min_cell_size=min_cell_size, variable_h=varh)
    cs = particles.cell_manager.cell_size
    kernel = base.CubicSplineKernel(dim=dim)
    for nm in ("o0", "o1", "o2"):
        f.add_property({"name": nm})
    types = [Fluid, Solid][:len(arrays)]
    refs = [to_oracle(a, k) for k, a in enumerate(arrays)]
    op = solver.SPHOperation(sph.SPHRho.withargs(), on_types=[Fluid], from_types=types,
                             updates=["rho"], id="rho")
    op.get_calcs(particles, kernel)[0].sph("o0")
    ref = O.sphrho(dim, refs[0], refs, cell_size=cs)
    assert max_rel(f.get("o0"), ref) < 1e-12
    ups = ["u", "v", "w"][:dim]
    op = solver.SPHIntegration(sph.MomentumEquation.withargs(alpha=0.5, beta=0.5, eta=0.1,
                                                             dim=dim),
                               on_types=[Fluid], from_types=types, updates=ups, id="mom")
    op.get_calcs(particles, kernel)[0].sph(*["o0", "o1", "o2"][:dim])
    got = np.stack([f.get(nm) for nm in ["o0", "o1", "o2"][:dim]])
    ref = O.momentum(dim, refs[0], refs, alpha=0.5, beta=0.5, eta=0.1, cell_size=cs)[:dim]
    if np.linalg.norm(ref) > 0:
        assert rel_norm(got, ref) < 1e-12
    else:
        assert not got.any()


@pytest.mark.parametrize("n", [1, 3, 4, 5, 63, 64, 65, 255, 257])
@pytest.mark.parametrize("dim", [2, 3])
def test_small_counts(n, dim):
    _check([_points(n, dim, 0.1, n, Fluid)], dim)


@pytest.mark.parametrize("n", [(1 << 14) - 1, 1 << 14, (1 << 15) - 1, 1 << 15])
def test_counts_where_the_lanes_change(n):
    h = 0.5 * (20 / (np.pi * n)) ** 0.5
    _check([_points(n, 2, h, 1, Fluid), _points(n // 3, 2, h, 2, Solid)], 2)


@pytest.mark.parametrize("n,dim,h", [(3000, 2, 0.15), (3000, 3, 0.25), (17000, 2, 0.05)])
def test_more_neighbours_than_the_queue_holds(n, dim, h):
    # 200 to 700 neighbours per particle; the queues hold 256 (128 from 16k
    # particles on)
    _check([_points(n, dim, h, 5, Fluid)], dim)


@pytest.mark.parametrize("n", [700, 17000])
def test_more_rows_than_the_list_holds(n):
    # search radius of 7 cells, 14 bins: up to 29 x 29 rows, lists of 128 / 64
    h = 0.14 if n < 1000 else 0.035
    _check([_points(n, 3, h, 6, Fluid)], 3, min_cell_size=2 * h / 7)


def test_points_beyond_the_cull_take_the_whole_ring():
    # 1e31: outside the range the FP32 cull is used in; the cells, the test
    # and the sums are FP64
    a = _points(200, 2, 1e30, 7, Fluid, spread=1e31)
    a.set(m=np.full(200, 1e60))
    particles = base.Particles([a])
    kernel = base.CubicSplineKernel(dim=2)
    op = solver.SPHOperation(sph.SPHRho.withargs(), on_types=[Fluid], from_types=[Fluid],
                             updates=["rho"], id="rho")
    op.get_calcs(particles, kernel)[0].sph("rho")
    ref = O.sphrho(2, to_oracle(a), [to_oracle(a)],
                   cell_size=particles.cell_manager.cell_size)
    assert max_rel(a.get("rho"), ref) < 1e-12


def test_mixed_radii_symmetric():
    a = _points(5000, 2, 0.01, 8, Fluid)
    rng = np.random.Generator(np.random.PCG64(9))
    a.set(h=0.01 * (1 + 4 * rng.random(5000) ** 4))
    particles = base.Particles([a], variable_h=True)
    kernel = base.CubicSplineKernel(dim=2)
    op = solver.SPHOperation(sph.SPHRho.withargs(), on_types=[Fluid], from_types=[Fluid],
                             updates=["rho"], id="rho")
    op.get_calcs(particles, kernel)[0].sph("rho")
    # every pair within the larger of the two radii, brute force
    x, y, h, m = (a.get(c) for c in ("x", "y", "h", "m"))
    r = np.sqrt((x[:, None] - x) ** 2 + (y[:, None] - y) ** 2)
    hab = 0.5 * (h[:, None] + h)
    q = r / hab
    w = 10.0 / (7.0 * np.pi * hab ** 2) * np.where(
        q > 2, 0.0, np.where(q > 1, 0.25 * (2 - q) ** 3, 1 - 1.5 * q * q * (1 - 0.5 * q)))
    w[r >= 2 * np.maximum(h[:, None], h)] = 0.0
    assert max_rel(a.get("rho"), (m * w).sum(1)) < 1e-12


def test_fp64_stage_2_on_the_stage_1_binning_counts_jumps_at_the_predictor():
    """RK2 in FP64 keeps the stage-1 binning in stage 2.  A particle whose
    predictor X1 lies more than one cell away is counted as the re-binning by
    X1 counted it, and the sums at X1 equal those of a re-binned stage 2
    (other order of the sums: 1e-12)."""
    from pysph_amd._abi import JumpToleranceError
    from pysph_amd.solver import generators as gen
    out = []
    for rebin in (False, True):
        f, _, info = gen.elliptical_drop_2d(2000, precision="double")
        particles = base.Particles([f])
        s = solver.wcsph_solver(2, co=info["co"], ro=1.0, alpha=0.1, with_solid=False)
        s.setup_integrator(particles)
        s.integrator.plan.stage2_rebin = rebin
        s.set_time_step(info["dt"])
        s.set_final_time(info["dt"] * 5.5)
        s.solve()
        out.append([f.get(c) for c in ("x", "y", "u", "v", "rho", "p")])
        u = f.get("u")
        u[7] = 5.0 * particles.cell_manager.cell_size / info["dt"]
        f.set(u=u)
        with pytest.raises(JumpToleranceError):
            for _ in range(2):
                s.integrator.integrate(info["dt"])
            particles.cell_manager.verify_jumps()
    for a, b in zip(*out):
        assert rel_norm(a, b) < 1e-12


@pytest.mark.parametrize("use_graph", [False, True])
def test_fp64_steps_with_a_fast_particle_rebin_in_stage_2(use_graph):
    """A particle that moves 0.3 cells a step, alone above the others: the
    steps re-bin in stage 2 instead of widening every stencil by its move,
    keep the stage-1 binning again some steps after it has slowed down, and
    agree with steps that always re-bin (other order of the sums: 1e-12)."""
    from pysph_amd.solver import generators as gen
    out = []
    for rebin in (False, True):
        f, _, info = gen.elliptical_drop_2d(2000, precision="double")
        particles = base.Particles([f])
        cm = particles.cell_manager
        s = solver.wcsph_solver(2, co=info["co"], ro=1.0, alpha=0.1, with_solid=False)
        s.setup_integrator(particles)
        plan = s.integrator.plan
        plan.stage2_rebin, plan.use_graph = rebin, use_graph

        def steps(k):
            n0, r0 = cm.num_binnings, plan.graph_replays
            for _ in range(k):
                s.integrator.integrate(info["dt"])
                torch.cuda.synchronize()
            return (cm.num_binnings - n0) / k, plan.graph_replays - r0

        steps(4)
        x, y, u, v = (f.get(c) for c in ("x", "y", "u", "v"))
        x[7], y[7], u[7], v[7] = 0.0, y.max() + 50 * cm.cell_size, \
            0.3 * cm.cell_size / info["dt"], 0.0
        f.set(x=x, y=y, u=u, v=v)
        cm.verify_jumps = lambda: 0
        cm._jump_seen = 1 << 30  # the particle was put there
        steps(6)
        per, replays = steps(20)
        if not rebin:
            assert not plan._keeps_binning() and cm.last_move > 0.25 * cm.cell_size
        if use_graph:
            assert replays > 0 and plan.graph_error is None
        else:
            assert per == 2
        u = f.get("u")
        u[7] = 0.0
        f.set(u=u)
        steps(plan.FAR_STEPS + 12)
        per, _ = steps(4)
        if not rebin:
            assert plan._keeps_binning() and cm.last_move < 0.1 * cm.cell_size
        if not use_graph:
            assert per == (2 if rebin else 1)
        out.append([f.get(c) for c in ("x", "y", "u", "v", "rho", "p")])
    for a, b in zip(*out):
        assert rel_norm(a, b) < 1e-12


@pytest.mark.parametrize("n,dim,h", [(1, 2, 0.1), (65, 3, 0.2), (3000, 2, 0.15), (3000, 3, 0.25),
                                     (17000, 2, 0.06), (17000, 3, 0.03)])
@pytest.mark.parametrize("shuffled", [False, True])
def test_row_fill_sorts_short_and_long_rows(n, dim, h, shuffled):
    """Rows that fit a group's share of LDS (128 entries; 256 below 16k
    particles) and rows that outgrow it, in user order, ascending but for the
    particle itself: the sets are whole numbers and must be equal."""
    a = _points(n, dim, h, 11, Fluid)
    if shuffled:
        # a first binning makes slot order and user order differ
        base.Particles([a]).cell_manager.update()
    particles = base.Particles([a])
    off, nb = particles.nnps_manager.get_neighbor_particle_locator(a, a, 2.0).get_csr()
    off_o, nb_o = O.nnps_csr(to_oracle(a), radius_scale=2.0,
                             cell_size=particles.cell_manager.cell_size)
    assert np.array_equal(off, off_o)
    for i in range(n):
        row = nb[off[i]:off[i + 1]]
        ref = np.sort(nb_o[off_o[i]:off_o[i + 1]])
        # the own index and the last entry change places (nnps.pyx:612-618)
        at = np.flatnonzero(ref == i)[0]
        ref[at], ref[-1] = ref[-1], i
        assert np.array_equal(row, ref)
    # without the own index moved
    from pysph_amd.base.nnps import neighbor_csr
    off2, nb2 = neighbor_csr(particles.cell_manager, a, a, 2.0)
    assert np.array_equal(off2, off)
    assert all(np.all(np.diff(nb2[off2[i]:off2[i + 1]]) > 0) for i in range(n))


@pytest.mark.parametrize("n,dim,h", [(65, 3, 0.2), (3000, 2, 0.15), (3000, 3, 0.25),
                                     (17000, 3, 0.06), ((1 << 17) + 5, 2, 0.0045)])
@pytest.mark.parametrize("kind", ["varh", "periodic"])
@pytest.mark.parametrize("ascending", [False, True])
def test_row_fill_of_symmetric_and_periodic_rows(n, dim, h, kind, ascending):
    """Short rows and rows of several hundred entries of the symmetric
    variable-h sets and of periodic ones (whose walk order is not ascending),
    with user ids and with slot ids, which are found in order: the oracle's
    sets, sorted."""
    from pysph_amd import _abi
    from pysph_amd._device import require_gpu
    a = _points(n, dim, h, 12, Fluid)
    rng = np.random.Generator(np.random.PCG64(3))
    if kind == "varh":
        a.set(h=h * (0.6 + 0.8 * rng.random(n)))
    dom = None
    if kind == "periodic":
        if 4 * h >= 1:
            pytest.skip("the box holds less than two search radii")
        dom = base.PeriodicDomain(xmin=0.0, xmax=1.0, ymin=0.0, ymax=1.0)
    particles = base.Particles([a], variable_h=kind == "varh", periodic_domain=dom)
    cm = particles.cell_manager
    cm.update()
    ao = to_oracle(a)
    if kind == "periodic":
        ext, origin = O.with_ghosts(ao, (1.0, 1.0, 0.0), (0.0, 0.0, 0.0), cm.cell_size,
                                    cm.cell_size)
        off_o, nb_o = O.nnps_csr(ao, ext, radius_scale=2.0, cell_size=cm.cell_size)
        nb_o = origin[nb_o]
    else:
        off_o, nb_o = O.nnps_csr(ao, radius_scale=2.0, varh=True)
    stream = require_gpu(a.get_carray("x"))
    v = a.view()
    slots = torch.arange(n, dtype=torch.int64, device=a.device)
    order = slots if a._order is None else a._order
    ids = slots if ascending else order
    counts = torch.empty(n, dtype=torch.int64, device=a.device)
    off = torch.empty(n + 1, dtype=torch.int64, device=a.device)
    total = _abi.ctypes.c_int64(0)
    rmax = 2.0 * cm.max_h if kind == "varh" else 0.0
    _abi.call("sph_neighbor_row_counts", stream, cm.grid, v, v, 2.0, rmax, order.data_ptr(),
              counts.data_ptr())
    _abi.call("sph_scan_counts", stream, n, counts.data_ptr(), off.data_ptr(),
              _abi.ctypes.byref(total))
    nbr = torch.empty(total.value, dtype=torch.int64, device=a.device)
    _abi.call("sph_neighbor_row_fill", stream, cm.grid, v, v, 2.0, rmax, order.data_ptr(),
              ids.data_ptr(), off.data_ptr(), nbr.data_ptr(), total.value, total.value, 0)
    assert np.array_equal(off.cpu().numpy(), off_o)
    nb = nbr.cpu().numpy()
    rows = np.repeat(np.arange(n), np.diff(off_o))
    inside = rows[1:] == rows[:-1]
    assert (nb[1:] > nb[:-1])[inside].all()
    users = order.cpu().numpy()[nb] if ascending else nb
    key = np.lexsort((users, rows))
    ref = np.lexsort((nb_o, rows))
    assert np.array_equal(users[key], nb_o[ref])
