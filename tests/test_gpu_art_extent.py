"""ART diffuse transfer on a long box whose extent along one axis is not its
cells' (a side face puts a ray back on the box's face, so every wrap shifts it):
the layer sweep below its bound and the launch per ray group above it both
equal the oracle."""
import numpy as np
import pytest

import oracle as O
from argot_amd import art as A
from argot_amd import radiation as R
from test_gpu_art_sweep import box

pytestmark = pytest.mark.gpu


# 400 layers wrap the z-dominant rays (slopes of 0.79) up to 10 times along the
# 34 cells of x, which are two tiles; extents off by just below and just above
# the sweep's bound (0.14 cells over all wraps, beside 0.06 for rounding), and by
# 0.4 cells over all wraps.  (Rays of a group, two cells apart, still share no cell.)
@pytest.mark.parametrize("off", [0.0098, 0.0108, 0.045])
@pytest.mark.parametrize("wider", [True, False])
def test_extent_off_the_cells(require_gpu, monkeypatch, off, wider):
    shape = (34, 64, 400)
    print(f"art extent off by {off} cells, wider {wider}", flush=True)
    w = box(shape, seed=77)
    h = float(np.float32(1.0) / np.float32(max(shape)))
    hi = [float(np.float32(k * h)) for k in shape]
    hi[0] = float(np.float32((shape[0] + (off if wider else -off)) * h))
    plain = R.run_param_for

    def run_param(*args):
        r = plain(*args)
        r.delta_x = r.delta_y = r.delta_z = h
        r.xmax, r.ymax, r.zmax = hi
        r.xmax_local, r.ymax_local, r.zmax_local = hi
        return r

    g = O.art_grid(max(shape), w.lunit, w.denstonh, w.helium_fact)
    g.nx, g.ny, g.nz = shape
    g.xmax, g.ymax, g.zmax = hi
    monkeypatch.setattr(R, "run_param_for", run_param)
    st = A.DiffuseStep(w, nside=1)
    stats = st.step()
    got = st.rates()
    st.close()
    ref, ncross = O.art_run(g, 1, w.dens, A.chem_array(w), A.UENETOK, True)
    assert stats["ncross"] == ncross
    floor = 1e-6 * np.abs(ref).max(0)
    err = np.abs(got.astype(np.float64) - ref) / np.maximum(np.abs(ref), floor)
    assert err.max() < 1e-5, err.max(0)
