"""ART diffuse transfer on boxes that the layer sweep splits into tiles, whose
axes differ, or whose coordinates are too coarse for it (a launch per ray
group then): rates and crossings equal the oracle's."""
import dataclasses

import numpy as np
import pytest

import oracle as O
from argot_amd import art as A
from argot_amd import ic
from argot_amd import radiation as R

pytestmark = pytest.mark.gpu


def compare(w, run_param, monkeypatch, g, batch, exp64):
    monkeypatch.setattr(R, "run_param_for", run_param)
    st = A.DiffuseStep(w, nside=2, batch=batch, exp64=exp64)
    stats = st.step()
    got = st.rates()
    st.close()
    ref, ncross = O.art_run(g, 2, w.dens, A.chem_array(w), A.UENETOK, True)
    assert stats["ncross"] == ncross
    assert np.isfinite(got).all()
    floor = 1e-6 * np.abs(ref).max(0)
    err = np.abs(got.astype(np.float64) - ref) / np.maximum(np.abs(ref), floor)
    assert err.max() < 1e-5, err.max(0)


def box(shape, seed):
    w = ic.art128(seed=seed, n=max(shape))
    cut = tuple(slice(0, k) for k in shape)
    fields = {f: np.ascontiguousarray(getattr(w, f)[cut])
              for f in ("dens", "fHI", "fHII", "fHeI", "fHeII", "fHeIII", "temper")
              if hasattr(w, f)}
    return dataclasses.replace(w, **fields)


# one tile and just past it, tiles along either axis and both, short last
# tiles, the smallest even axes
@pytest.mark.parametrize("shape", [(64, 64, 2), (66, 66, 4), (4, 128, 66), (130, 6, 70),
                                   (2, 2, 200), (68, 72, 96), (6, 4, 600), (40, 12, 300)])
@pytest.mark.parametrize("exp64", [False, True])
def test_tiled_sweep_matches_oracle(require_gpu, monkeypatch, shape, exp64):
    print(f"art sweep {shape} exp64={exp64}", flush=True)
    w = box(shape, seed=sum(shape))
    h = float(np.float32(1.0) / np.float32(max(shape)))
    hi = [float(np.float32(k * h)) for k in shape]
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
    compare(w, run_param, monkeypatch, g, 20, exp64)


@pytest.mark.parametrize("lo", [500.0, 1500.0, -4000.0])   # below and above the sweep's bound
@pytest.mark.parametrize("exp64", [False, True])
def test_far_box_matches_oracle(require_gpu, monkeypatch, lo, exp64):
    print(f"art far box {lo} exp64={exp64}", flush=True)
    w = ic.art128(seed=31, n=16)
    hi = lo + 1.0
    plain = R.run_param_for

    def run_param(*args):
        r = plain(*args)
        r.xmin = r.ymin = r.zmin = r.xmin_local = r.ymin_local = r.zmin_local = lo
        r.xmax = r.ymax = r.zmax = r.xmax_local = r.ymax_local = r.zmax_local = hi
        return r

    g = O.art_grid(16, w.lunit, w.denstonh, w.helium_fact, lo, hi)
    compare(w, run_param, monkeypatch, g, 0, exp64)
