"""What a replayed step looks up on the host: the reduced bounds rows, and
the key of the live arrays against that of a recorded state."""
import itertools

import numpy as np
import pytest

from pysph_amd.base.cell import CellManager
from pysph_amd.base.particle_array import get_particle_array
from pysph_amd.base.step_graph import StepGraphs

INF, NAN = np.inf, np.nan


@pytest.mark.parametrize("odd", [None, INF, -INF, NAN])
def test_bounds_rows_reduce_like_arrays(odd):
    rng = np.random.Generator(np.random.PCG64(3))
    rows = rng.normal(0, 1, (3, 8))
    for r, c in itertools.product(range(3), range(7)):
        b = rows.copy()
        if odd is not None:
            b[r, c] = odd
        lo, hi, hm = CellManager._reduce_bounds(b)
        with np.errstate(invalid="ignore"):
            wl, wh, wm = b[:, :3].min(0), b[:, 3:6].max(0), b[:, 6].max()
        bad = ~(np.isfinite(wl) & np.isfinite(wh))
        wl[bad] = wh[bad] = 0
        assert list(lo) == list(wl) and list(hi) == list(wh)
        assert hm == wm or (np.isnan(hm) and np.isnan(wm))


class _Cells:
    grid, is_dirty = None, True


def test_live_key_is_the_key_of_the_state():
    pas = [get_particle_array(name=n, x=np.zeros(k)) for n, k in (("a", 3), ("b", 2))]
    sg = StepGraphs(pas, _Cells(), key_extra=lambda: (1, 2))
    k0 = sg.live_key()
    assert k0 == sg.key(sg.state())
    # the order of the properties is no part of it, their buffers are
    p = pas[0]._props
    x = p.pop("x")
    assert sg.live_key() != k0
    p["x"] = x
    assert sg.live_key() == k0 == sg.key(sg.state())
    p["x"] = x.clone()
    assert sg.live_key() != k0
    p["x"] = x
    pas[1].set_dirty(not pas[1].is_dirty)
    assert sg.live_key() != k0 and sg.live_key() == sg.key(sg.state())
