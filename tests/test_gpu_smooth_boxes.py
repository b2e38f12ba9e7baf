"""Smoothing on boxes whose axes are not multiples of the kernel's tiles equals
the oracle's bit for bit, on the device and in the host mesh."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

import oracle as O
from argot_amd import abi
from argot_amd import radiation as R
from argot_amd._lib import lib
from helpers import small_workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(4, 4, 16), (5, 3, 70), (1, 1, 2), (2, 17, 1), (7, 130, 33)])
def test_smoothing_matches_oracle(require_gpu, shape):
    print(f"smooth {shape}", flush=True)
    n = int(np.prod(shape))
    w = small_workload(n=16, nsrc=1, seed=9)
    rng = np.random.default_rng(n)
    cells = rng.integers(0, w.dens.size, n)
    w = dataclasses.replace(w, **{f: np.ascontiguousarray(
        np.asarray(getattr(w, f)).reshape(-1)[cells].reshape(shape))
        for f in ("dens", "fHI", "fHII", "fHeI", "fHeII", "fHeIII")})
    st = R.PointSourceStep(w)
    raw = (rng.random((n, 6)) * 10.0 ** rng.integers(-20, -10, (n, 6))).astype(np.float32)
    v = abi.mesh_view(st.mesh)
    pc = v["prev_chem"]
    for k, f in enumerate(R.RATE_FIELDS):
        pc[f] = raw[:, k]
    v["prev_chem"] = pc
    lib().zero_out_photoion_rate_cuda(C.byref(st.cmem), C.byref(st.cpar), C.byref(st.run))
    lib().merge_photoion_data(st.mesh, C.byref(st.cmem), C.byref(st.cpar), C.byref(st.run))
    st.smooth()
    host = np.stack([abi.mesh_view(st.mesh)["prev_chem"][f] for f in R.RATE_FIELDS], axis=1)
    ref = O.smooth_rates(raw, shape)
    np.testing.assert_array_equal(host, ref)
    np.testing.assert_array_equal(st.rates(), ref)
