"""The SoA passes and neighbour counts where large sets leave the groups of lanes: one lane per
destination from 2^15 particles on in 1D and 2^18 in 2D (2^17 with two
sources, 2^19 with periodic axes), fewer lanes from 2^17 (2D) and 2^20 (3D) on, against the FP64 oracle on the same stored bits; plain,
periodic and symmetric variable-h sets.  FP64 within 1e-12 (sums of at most
1e3 terms, as in test_gpu_group.py)."""
import numpy as np
import pytest
import torch

import pysph_amd.base.api as base
import pysph_amd.solver.api as solver
import pysph_amd.sph.api as sph
from oracle import oracle as O
from pysph_amd import _abi
from pysph_amd._device import require_gpu
from tests.util import rel_norm, to_oracle

pytestmark = pytest.mark.gpu
Fluid = base.ParticleType.Fluid
Solid = base.ParticleType.Solid


def _set(n, dim, nbrs, seed, vary=0.0, precision="double"):
    rng = np.random.Generator(np.random.PCG64(seed))
    pos = rng.random((3, n))
    vel = rng.normal(size=(3, n))
    pos[dim:] = 0.0
    vel[dim:] = 0.0
    vol = {1: 2.0, 2: np.pi, 3: 4.0 / 3.0 * np.pi}[dim]
    h = 0.5 * (nbrs / (vol * n)) ** (1.0 / dim)
    return base.get_particle_array(
        name="s", type=Fluid, cl_precision=precision, x=pos[0], y=pos[1], z=pos[2], u=vel[0], v=vel[1], w=vel[2],
        h=h * (1.0 + vary * rng.random(n)), m=0.5 + rng.random(n),
        rho=1000.0 + 10 * rng.random(n), p=1e3 * rng.random(n), cs=10.0 + rng.random(n))


@pytest.fixture(autouse=True)
def _oracle_threads():
    O.set_threads(0)
    yield
    O.set_threads(1)


@pytest.mark.parametrize("n,dim,kind", [
    ((1 << 17) - 1, 2, "plain"), (1 << 17, 2, "plain"), ((1 << 18) - 1, 2, "plain"),
    (1 << 18, 2, "plain"), (1 << 18, 2, "periodic"), (1 << 18, 2, "varh"),
    ((1 << 15) - 1, 1, "plain"), (1 << 15, 1, "plain"), (1 << 15, 1, "periodic"),
    (1 << 15, 1, "varh"), ((1 << 17) - 1, 2, "two"), (1 << 17, 2, "two"), (1 << 19, 2, "periodic"),
    (1 << 20, 3, "plain")])
def test_sums_where_the_lanes_change(n, dim, kind):
    a = _set(n, dim, 15, 3, 0.5 if kind == "varh" else 0.0)
    dom = None
    if kind == "periodic":
        dom = base.PeriodicDomain(xmin=0.0, xmax=1.0,
                                  **({} if dim == 1 else dict(ymin=0.0, ymax=1.0)))
    b = [_set(n // 3, dim, 15, 4)] if kind == "two" else []
    for pa in b:
        pa.set(h=np.full(n // 3, a.get("h")[0]))
        pa.particle_type = Solid
    particles = base.Particles([a] + b, variable_h=kind == "varh", periodic_domain=dom)
    cs = particles.cell_manager.cell_size
    kernel = base.CubicSplineKernel(dim=dim)
    for nm in ("o0", "o1", "o2"):
        a.add_property({"name": nm})
    ao = to_oracle(a)
    src = [ao] + [to_oracle(pa, 1) for pa in b]
    if kind == "periodic":
        src[0], _ = O.with_ghosts(ao, (1.0, 1.0 if dim > 1 else 0.0, 0.0), (0.0, 0.0, 0.0), cs,
                                  cs)
    kw = dict(cell_size=cs, varh=kind == "varh")
    F, G = [Fluid], [Solid] if b else []
    op = solver.SPHOperation(sph.SPHRho.withargs(), on_types=F, from_types=F + G, updates=["rho"],
                             id="rho")
    op.get_calcs(particles, kernel)[0].sph("o0")
    assert rel_norm(a.get("o0"), O.sphrho(dim, ao, src, **kw)) < 1e-12
    op = solver.SPHIntegration(sph.SPHDensityRate.withargs(hks=False), on_types=F, from_types=F + G,
                               updates=["rho"], id="rate")
    op.get_calcs(particles, kernel)[0].sph("o0")
    assert rel_norm(a.get("o0"), O.density_rate(dim, ao, src, **kw)) < 1e-12
    op = solver.SPHIntegration(sph.MomentumEquation.withargs(alpha=0.5, beta=0.5, eta=0.1,
                                                             dim=dim),
                               on_types=F, from_types=F + G, updates=["u", "v", "w"][:dim], id="mom")
    op.get_calcs(particles, kernel)[0].sph(*["o0", "o1", "o2"][:dim])
    got = np.stack([a.get(nm) for nm in ["o0", "o1", "o2"][:dim]])
    ref = O.momentum(dim, ao, src, alpha=0.5, beta=0.5, eta=0.1, **kw)[:dim]
    assert rel_norm(got, ref) < 1e-12


@pytest.mark.parametrize("n,dim,kind,precision", [
    ((1 << 17) - 1, 2, "plain", "single"), (1 << 17, 2, "plain", "single"),
    (1 << 17, 2, "plain", "double"), (1 << 17, 2, "periodic", "single"),
    (1 << 17, 2, "varh", "double"), ((1 << 15) - 1, 1, "plain", "double"),
    (1 << 15, 1, "plain", "double"), (1 << 15, 1, "periodic", "double"), ((1 << 19) - 1, 3, "plain", "single"),
    (1 << 19, 3, "plain", "single"), (1 << 19, 3, "plain", "double")])
@pytest.mark.parametrize("bins", [1, 2])
def test_counts_where_the_lanes_change(n, dim, kind, precision, bins):
    """Neighbour counts are whole numbers: equal to the oracle's."""
    a = _set(n, dim, 15, 5, 0.5 if kind == "varh" else 0.0, precision)
    dom = None
    if kind == "periodic":
        dom = base.PeriodicDomain(xmin=0.0, xmax=1.0,
                                  **({} if dim == 1 else dict(ymin=0.0, ymax=1.0)))
    particles = base.Particles([a], variable_h=kind == "varh", periodic_domain=dom)
    cm = particles.cell_manager
    cm.set_cells_per_radius(bins)
    cm.update()
    ao = to_oracle(a)
    src = ao
    if kind == "periodic":
        src, _ = O.with_ghosts(ao, (1.0, 1.0 if dim > 1 else 0.0, 0.0), (0.0, 0.0, 0.0),
                               cm.cell_size, cm.cell_size)
    off, _ = O.nnps_csr(ao, src, cell_size=cm.cell_size, varh=kind == "varh")
    v = a.view()
    counts = torch.empty(n, dtype=torch.int64, device=a.device)
    _abi.call("sph_neighbor_row_counts", require_gpu(counts), cm.grid, v, v, 2.0,
              2.0 * cm.max_h if kind == "varh" else 0.0, a._order.data_ptr(), counts.data_ptr())
    assert np.array_equal(counts.cpu().numpy(), np.diff(off))
