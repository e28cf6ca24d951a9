"""sph_bin and sph_bounds against numpy on the same stored values, at the
sizes where the single-block binning (up to 8192 particles and 32767 cells)
hands over to the general path, with particles outside the grid and NaN.
Cells, permutations and extrema are whole numbers or copies: equal exactly."""
import numpy as np
import pytest
import torch

from pysph_amd import _abi
from pysph_amd._device import require_gpu

pytestmark = pytest.mark.gpu


def _view(pos, h):
    v = _abi.SphView()
    v.n = len(h)
    v.dtype = _abi.SPH_F32 if h.dtype == torch.float32 else _abi.SPH_F64
    v.x, v.y, v.z, v.h = (t.data_ptr() for t in pos + [h])
    return v


def _points(n, dtype, seed, lo=-0.5, hi=1.5):
    rng = np.random.Generator(np.random.PCG64(seed))
    p = rng.uniform(lo, hi, (3, n)).astype(np.float32 if dtype == torch.float32 else np.float64)
    return p, [torch.from_numpy(a).cuda() for a in p]


@pytest.mark.parametrize("n", [1, 2, 1023, 1024, 1025, 8191, 8192, 8193])
@pytest.mark.parametrize("dims", [(1, 1, 1), (31, 32, 33), (32767, 1, 1), (32, 32, 32), (7, 5, 3)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_bin_is_the_stable_sort_by_cell(n, dims, dtype):
    p, pos = _points(n, dtype, n)
    if n > 4:
        pos[0][3] = float("nan")
        p[0][3] = np.nan
    h = torch.ones(n, dtype=dtype, device="cuda")
    g = _abi.SphGrid()
    g.cell_size = 1.0 / max(dims)
    for d in range(3):
        g.lo[d], g.dims[d] = 0, dims[d]
    nc = dims[0] * dims[1] * dims[2]
    ws = torch.empty(_abi.load().sph_bin_workspace_bytes(n, nc), dtype=torch.uint8, device="cuda")
    perm, cell, start = (torch.empty(k, dtype=torch.int32, device="cuda") for k in (n, n, nc + 1))
    # previous cells: every second particle two bins away in x where there is room
    with np.errstate(invalid="ignore"):
        c = [np.floor(a.astype(np.float64) / g.cell_size) for a in p]
    c = [np.where(np.isnan(a), 0, np.clip(a, 0, k - 1)).astype(np.int64) for a, k in zip(c, dims)]
    key = (c[2] * dims[1] + c[1]) * dims[0] + c[0]
    px = np.where(np.arange(n) % 2 == 0, c[0], (c[0] + 2) % dims[0])
    prev = torch.from_numpy(((c[2] * dims[1] + c[1]) * dims[0] + px).astype(np.int32)).cuda()
    jumps = torch.zeros(1, dtype=torch.int32, device="cuda")
    _abi.call("sph_bin", require_gpu(perm), _view(pos, h), g, perm.data_ptr(), cell.data_ptr(),
              start.data_ptr(), prev.data_ptr(), jumps.data_ptr(), ws.data_ptr(), ws.numel())
    order = np.argsort(key, kind="stable")
    assert np.array_equal(perm.cpu().numpy(), order)
    assert np.array_equal(cell.cpu().numpy(), key[order])
    assert np.array_equal(start.cpu().numpy(), np.searchsorted(key[order], np.arange(nc + 1)))
    assert int(jumps.item()) == int((np.abs(px - c[0]) > 1).sum())


@pytest.mark.parametrize("n", [1, 63, 1025, 4 * 65536 - 1, 4 * 65536 + 1, 600011])
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
def test_bounds_are_the_extrema(n, dtype):
    p, pos = _points(n, dtype, n + 7)
    if n > 100:
        p[1][17] = np.nan
        pos[1][17] = float("nan")
    h = torch.from_numpy(np.abs(p[2]) + 0.1).to(dtype).cuda()
    out = torch.empty(_abi.SPH_BOUNDS_WORDS, dtype=torch.float64, device="cuda")
    _abi.call("sph_bounds", require_gpu(out), _view(pos, h), out.data_ptr())
    got = out[:7].cpu().numpy()
    want = [np.nanmin(a) for a in p] + [np.nanmax(a) for a in p] + [float(h.max())]
    assert np.array_equal(got, np.array(want, dtype=np.float64))
