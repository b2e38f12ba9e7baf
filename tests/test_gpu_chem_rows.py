"""Cells with many sub-steps, which the chemistry hands from its one-lane
kernel to rows of 16 lanes: the same bits, counts and maxima as the kernel
that gives every cell one thread, with none, a few, and more of them than the
hand-over list holds (16384), among them cells at both energy bounds, at the
980 K break and cells that turn NaN."""
import numpy as np
import pytest

from argot_amd import abi, ic
from argot_amd import radiation as R
from argot_amd._lib import lib
from helpers import small_workload

pytestmark = pytest.mark.gpu


def mesh_step(n, seed, share, gamma):
    w = small_workload(n=n, nsrc=1, seed=seed)
    st = R.PointSourceStep(w)
    v = abi.mesh_view(st.mesh)
    ncell = n ** 3
    rng = np.random.default_rng(seed)
    strong = rng.random(ncell) < share
    g = np.where(strong, gamma * 10.0 ** rng.uniform(-0.5, 0.5, ncell), 1e-17)
    pc = v["prev_chem"]
    for f, k in zip(R.RATE_FIELDS, (1.0, 1.6e-11, 0.9, 0.08, 2.0e-11, 4.0e-12)):
        pc[f] = (g * k).astype(np.float32)
    if share > 0:
        pc["GammaHI"][0] = np.inf        # a cell that holds a source
    t = 10.0 ** rng.uniform(1.0, 6.0, ncell)
    t[1:4] = (10.0, 979.9, 1.0e8)
    v["prev_chem"] = pc
    v["chem"] = pc
    uenetok = ic.chem_units(w.lunit, w.denstonh)["uenetok"]
    u = (t / (uenetok * pc["wmol"].astype(np.float64))).astype(np.float32)
    v["uene"] = u
    v["prev_uene"] = u
    st.send_mesh()
    return st


@pytest.mark.parametrize("n,share,gamma,dtime", [(8, 0.0, 0.0, 1e-6), (8, 0.02, 1e-10, 1e-3),
                                                 (12, 0.3, 1e-11, 1e-3), (32, 0.9, 1e-11, 2e-4)])
def test_rows_equal_one_cell_per_thread(require_gpu, n, share, gamma, dtime):
    L = lib()
    st = mesh_step(n, 81, share, gamma)
    ref = np.frombuffer(st.mesh, np.uint8).copy()
    try:
        L.argot_hip_set_chem_queue(0)
        d0 = st.chemistry(np.float32(dtime))
        c0 = st.chem_stats()
        m0 = st.mesh_bytes()
        np.copyto(np.frombuffer(st.mesh, np.uint8), ref)
        st.send_mesh()
        L.argot_hip_set_chem_queue(1)
        d1 = st.chemistry(np.float32(dtime))
        c1 = st.chem_stats()
        m1 = st.mesh_bytes()
    finally:
        L.argot_hip_set_chem_queue(1)
    if share > 0:
        assert c0["nsub"] > 64 * 0.5 * share * n ** 3
    assert np.array_equal(m0, m1)
    assert np.array_equal(d0, d1, equal_nan=True)
    for k in ("nsub", "niter", "nstopped"):
        assert c0[k] == c1[k], k
