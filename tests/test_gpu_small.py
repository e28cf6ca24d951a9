"""Groups of lanes sharing a destination in the packed FP32 passes: the same
bits as the scans of one lane per destination, at the sizes where the lane
count changes and where a group's queue or row list overflows.

The same particles are summed twice: alone, and as the first n slots of a
larger set whose other particles are far away (many search radii), so that
the larger set takes the scans.  A destination has the same sources in the
same order both times, so the sums must be equal bit for bit; and they must
match the FP64 oracle within the FP32 contract (1e-5, as in
test_gpu_passes.py)."""
import numpy as np
import pytest
import torch

import pysph_amd.base.api as base
from oracle import oracle as O
from pysph_amd import _abi
from pysph_amd.sph import _ops
from tests.util import max_rel, to_oracle

pytestmark = pytest.mark.gpu


def _set(n, dim, h, seed, far, vary_h):
    """n random particles in the unit box, and `far` more on a coarse lattice
    beyond x = 1 + 20 h."""
    rng = np.random.Generator(np.random.PCG64(seed))
    pos = rng.random((3, n))
    vel = rng.normal(size=(3, n))
    hh = h * (np.ones(n) + (0.3 * rng.random(n) if vary_h else 0.0))
    k = int(np.ceil(far ** (1.0 / dim))) if far else 0
    grid = np.stack(np.meshgrid(*[np.arange(k)] * dim, indexing="ij")).reshape(dim, -1)[:, :far]
    fp = np.zeros((3, far))
    fp[:dim] = grid * 2.2 * h
    fp[0] += 1.0 + 20.0 * h
    pos = np.concatenate([pos, fp], 1)
    vel = np.concatenate([vel, np.zeros((3, far))], 1)
    pos[dim:] = 0.0
    vel[dim:] = 0.0
    m = n + far
    mass = np.concatenate([0.5 + rng.random(n), np.ones(far)])
    rho = np.concatenate([1000.0 + 10 * rng.random(n), np.full(far, 1000.0)])
    p = np.concatenate([1e3 * rng.random(n), np.zeros(far)])
    cs = np.concatenate([10.0 + rng.random(n), np.full(far, 10.0)])
    return base.get_particle_array(
        cl_precision="single", name="s", x=pos[0], y=pos[1], z=pos[2], u=vel[0], v=vel[1],
        w=vel[2], h=np.concatenate([hh, np.full(far, h)]), m=mass, rho=rho, p=p, cs=cs), m


def _sums(pa, dim, bins, disp=None):
    cm = base.CellManager(arrays_to_bin=[pa])
    cm.check_jumps = False
    cm.set_cells_per_radius(bins)
    cm.update()
    n = pa.get_number_of_particles()
    prm = _ops.make_params(dim, co=10.0, ro=1000.0, alpha=0.5, beta=0.5, eps=0.5)
    ov = _ops.packed_override([pa])
    aux = torch.empty((n, 4), dtype=torch.float32, device=pa.device)
    ov[id(pa)]["aux4"] = aux
    mk = lambda: torch.empty(n, dtype=torch.float32, device=pa.device)  # noqa: E731
    rho, p, cs = mk(), mk(), mk()
    _ops.density(cm, prm, pa, [pa], rho, p, cs, override=ov, disp=disp)
    acc, dv = [mk() for _ in range(3)], [mk() for _ in range(3)]
    _ops.momentum_xsph(cm, prm, pa, [pa], [_abi.SPH_SRC_MOMENTUM | _abi.SPH_SRC_XSPH], acc=acc,
                       dv=dv, override=ov, disp=disp)
    out = []
    order = pa._order_np()
    for t in [rho, p, cs] + acc + dv:
        a = np.empty(n, dtype=np.float32)
        a[order] = t.cpu().numpy()
        out.append(a)
    return out, cm


@pytest.mark.parametrize("dim,n,h,bins", [
    (2, 1, 0.1, 2), (2, 7, 0.3, 2), (2, 65, 0.15, 2), (2, 3000, 0.02, 2), (2, 11999, 0.011, 2),
    (2, 12000, 0.011, 2), (2, 35999, 0.006, 2), (3, 17, 0.3, 2), (3, 7999, 0.04, 2),
    (3, 16000, 0.03, 2), (3, 31999, 0.025, 2),
    # more neighbours than the queue holds (256 a group), more rows (128)
    (2, 3000, 0.2, 2), (3, 3000, 0.25, 2), (3, 1500, 0.1, 7)])
@pytest.mark.parametrize("vary_h", [False, True])
def test_groups_give_the_bits_of_the_scans(dim, n, h, bins, vary_h):
    a, _ = _set(n, dim, h, 3, 0, vary_h)
    b, m = _set(n, dim, h, 3, 70000, vary_h)
    got, cm = _sums(a, dim, bins)
    ref, _ = _sums(b, dim, bins)
    for k, (x, y) in enumerate(zip(got, ref)):
        assert np.array_equal(x, y[:n]), (k, np.abs(x - y[:n]).max())
    rho = O.sphrho(dim, to_oracle(a), [to_oracle(a)], cell_size=cm.cell_size)
    assert max_rel(got[0], rho) < 1e-5


def test_groups_over_a_widened_stencil_give_the_same_bits():
    a, _ = _set(3000, 2, 0.02, 3, 0, False)
    got, _ = _sums(a, 2, 2)
    disp = torch.full((1,), 0.013, dtype=torch.float32, device=a.device)
    wide, _ = _sums(a, 2, 2, disp=disp)
    for x, y in zip(got, wide):
        assert np.array_equal(x, y)
