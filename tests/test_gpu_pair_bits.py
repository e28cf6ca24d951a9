"""The rounding of the packed FP32 pair arithmetic, pinned bit for bit.

|r|^2 is fma(z, z, fma(x, x, y * y)) and (v . r) is fma(vz, z, fma(vx, x,
vy * y)) in every packed kernel, and 2 - r / h is one fma where a source of
uniform h feeds both the momentum and the XSPH sum: results stay what they
were to the last bit when a kernel is rewritten.  The hardware's square root and reciprocals have
no host equivalent, so a pair is compared with another pair that gives the
same rounded |r|^2 (or v . r) from one component alone: everything after it
is the same arithmetic on the same bits."""
from fractions import Fraction

import numpy as np
import pytest
import torch

import pysph_amd.base.api as base
from pysph_amd import _abi
from pysph_amd.sph import _ops

pytestmark = pytest.mark.gpu
F = np.float32
# destinations from which the packed passes take one lane each (2D)
SCAN_MIN = {"density": 12000, "momentum": 36000}


def _fma(a, b, c):
    return F(float(Fraction(float(a)) * Fraction(float(b)) + Fraction(float(c))))


def _near(x):
    out = [F(x)]
    for d in (-np.inf, np.inf):
        y = F(x)
        for _ in range(3):
            y = np.nextafter(y, F(d))
            out.append(y)
    return out


def _samples(count, make):
    """make(rng) -> a sample or None."""
    rng = np.random.Generator(np.random.PCG64(17))
    out = []
    while len(out) < count:
        s = make(rng)
        if s is not None:
            out.append(s)
    return out


def _array(name, x, y, u, v, pad, h):
    """One particle at (x, y) and `pad` far ones, of smoothing length h (a
    tuple: those of the two kinds)."""
    k = int(np.ceil(np.sqrt(pad))) if pad else 0
    gx, gy = np.meshgrid(np.arange(k), np.arange(k))
    fx, fy = 100.0 + 5.0 * gx.ravel()[:pad], 100.0 + 5.0 * gy.ravel()[:pad]
    n = pad + 1
    hh = np.full(n, h[1])
    hh[0] = h[0]
    one = np.ones(n)
    vel = np.zeros((2, n))
    vel[:, 0] = u, v
    return base.get_particle_array(
        name=name, cl_precision="single", x=np.concatenate([[x], fx]),
        y=np.concatenate([[y], fy]), z=0 * one, u=vel[0], v=vel[1], w=0 * one, h=hh, m=one,
        rho=1000.0 * one, p=3.0 * one, cs=10.0 * one)


def _first(pa, t):
    a = t.cpu().numpy()
    o = pa._order_np()
    return a[0] if o is None else a[np.flatnonzero(o == 0)[0]]


def _pass(kind, src, uniform, pad, flags=_abi.SPH_SRC_MOMENTUM, h=1.0):
    """The first output(s) of a destination at the origin at rest, with the
    source particle src = (x, y, u, v) of roles `flags`."""
    D = _array("d", 0.0, 0.0, 0.0, 0.0, pad, (h, h))
    # one far source of another h: the source's h is not uniform then
    S = _array("s", *src, 0 if uniform else 1, (h, h if uniform else 0.9 * h))
    cm = base.CellManager(arrays_to_bin=[D, S])
    cm.check_jumps = False
    cm.update()
    prm = _ops.make_params(2, co=10.0, ro=1000.0, alpha=0.5, beta=0.5, eps=0.5)
    n = D.get_number_of_particles()
    mk = lambda: torch.empty(n, dtype=torch.float32, device=D.device)  # noqa: E731
    ov = _ops.packed_override([D, S])
    if kind == "density":
        rho = mk()
        _ops.density(cm, prm, D, [S], rho, override=ov)
        return [_first(D, rho)]
    for pa in (D, S):
        k = pa.get_number_of_particles()
        aux = torch.empty((k, 4), dtype=torch.float32, device=pa.device)
        aux[:] = torch.tensor([1000.0, 10.0, 3e-6, 3.0], device=pa.device)
        ov[id(pa)]["aux4"] = aux
    acc, dv = [mk() for _ in range(3)], [mk() for _ in range(3)]
    _ops.momentum_xsph(cm, prm, D, [S], [flags], acc=acc, dv=dv, override=ov)
    return [_first(D, t) for t in acc + dv]


def _square_of(v):
    return next((c for c in _near(np.sqrt(F(v))) if F(c * c) == v), None)


@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("groups", [True, False])
def test_squared_distance(groups, uniform):
    pad = 0 if groups else SCAN_MIN["density"]

    def make(rng):
        a, b = F(rng.uniform(0.3, 1.3)), F(rng.uniform(0.3, 1.3))
        mine, other = _fma(a, a, F(b * b)), _fma(b, b, F(a * a))
        c, d = _square_of(mine), _square_of(other)
        return None if mine == other or c is None or d is None else (a, b, c, d)
    told = 0
    for a, b, c, d in _samples(16, make):
        got = _pass("density", (a, b, 0, 0), uniform, pad)
        want = _pass("density", (c, 0, 0, 0), uniform, pad)
        assert got[0] > 0 and got == want, (a, b, got, want)
        told += want != _pass("density", (d, 0, 0, 0), uniform, pad)
    assert told >= 4  # the other rounding would have been seen


@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("groups", [True, False])
def test_velocity_product(groups, uniform):
    pad = 0 if groups else SCAN_MIN["momentum"]

    def make(rng):
        x, y, u, v = (F(rng.uniform(0.3, 1.2)) for _ in range(4))
        # r = (-x, -y), velocity difference (u, v) with source velocity
        # (-u, -v): approaching, the viscous term is on
        mine, other = _fma(u, x, F(v * y)), _fma(v, y, F(u * x))
        p = next((k for k in _near(mine / x) if F(k * x) == mine), None)
        q = next((k for k in _near(other / x) if F(k * x) == other), None)
        return None if mine == other or p is None or q is None else (x, y, u, v, p, q)
    told = 0
    for x, y, u, v, p, q in _samples(16, make):
        got = _pass("momentum", (x, y, -u, -v), uniform, pad)
        want = _pass("momentum", (x, y, -p, 0), uniform, pad)
        assert got[0] != 0 and got[:3] == want[:3], (x, y, u, v, got, want)
        told += want[:3] != _pass("momentum", (x, y, -q, 0), uniform, pad)[:3]
    assert told >= 4


@pytest.mark.parametrize("uniform", [True, False])
def test_roles_and_groups(uniform):
    """A pair's momentum and XSPH terms for a source of both roles, of one
    role, from groups of lanes and from one lane per destination.  Groups and
    scans agree bit for bit in every role.  With a uniform h that is no power
    of two, 2 - r / h of the outer gradient branch is one fma for a source of
    both roles and a rounded quotient for one of momentum alone: apart in some
    pairs, by what a half last bit of r / h below 2 is of (2 - r / h)^3 at the
    largest r / h, 3 * 2^-24 / (2 - 1.93) = 2.6e-6, and twice that of the other
    roundings beside it."""
    M, X = _abi.SPH_SRC_MOMENTUM, _abi.SPH_SRC_XSPH
    rng = np.random.Generator(np.random.PCG64(5))
    apart = 0
    for _ in range(24):
        a = rng.uniform(0, 2 * np.pi)
        r = rng.uniform(0.75, 1.35)  # q from 1.07 to 1.93
        src = (F(r * np.cos(a)), F(r * np.sin(a)), F(rng.uniform(-1, 1)), F(rng.uniform(-1, 1)))
        out = {}
        for flags in (M, X, M | X):
            out[flags] = _pass("momentum", src, uniform, 0, flags, 0.7)
            scan = _pass("momentum", src, uniform, SCAN_MIN["momentum"], flags, 0.7)
            assert out[flags] == scan, (flags, src)
        both, mom, xs = np.array(out[M | X]), np.array(out[M]), np.array(out[X])
        assert np.all(mom[3:] == 0) and np.all(xs[:3] == 0) and both[0] != 0 and both[3] != 0
        assert np.allclose(both[:3], mom[:3], rtol=5e-6, atol=0)
        assert np.allclose(both[3:], xs[3:], rtol=5e-6, atol=0)
        apart += np.any(both[:3] != mom[:3])
    assert apart >= 4 if uniform else apart == 0
