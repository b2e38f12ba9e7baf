"""Segment lists whose wavefronts take the walk's float form with caps of every
size (segments of no length to the whole of a long box, ends on faces and
corners), and lists where a few wavefronts meet an end outside the box: every
optical depth equals the oracle's."""
import ctypes as C

import numpy as np
import pytest

from argot_amd import abi
from argot_amd import radiation as R
from argot_amd._lib import check, lib
from helpers import oracle_problem, ragged_workload

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(16, 16, 16), (5, 260, 9), (12, 7, 20)])
@pytest.mark.parametrize("outside", [0, 1, 40])   # of 3037 segments
def test_segment_lists_equal_the_oracle(require_gpu, shape, outside):
    w = ragged_workload(shape, nsrc=2, seed=93)
    P = oracle_problem(w)
    step = R.PointSourceStep(w)
    rng = np.random.default_rng(94 + outside)
    n = 3037
    size = np.array(shape)
    s = rng.uniform(0.0, 1.0, (n, 3)).astype(np.float32)
    e = rng.uniform(0.0, 1.0, (n, 3)).astype(np.float32)
    # lengths over the logarithm of the range, and the box's diagonal
    e = (s + (e - s) * 10 ** rng.uniform(-3, 0, (n, 1))).astype(np.float32)
    s[::31], e[::31] = 0.0, 1.0
    face = (rng.integers(0, size + 1, (n, 3)) / size).astype(np.float32)
    on = rng.random((n, 3)) < 0.2
    e[on] = face[on]
    s[::23] = e[::23]
    out = rng.choice(n, outside, replace=False)
    e[out] = rng.choice(np.float32([-0.2, 1.2]), (outside, 3))
    print(f"walk caps {shape}, {outside} ends outside", flush=True)
    segp = C.c_void_p()
    L = lib()
    L.allocate_pinned_segment(C.byref(segp), n)
    check("allocate_pinned_segment")
    try:
        seg = abi.view_at(abi.RaySegment, segp.value, n)
        for k, a in enumerate("xyz"):
            seg[f"{a}pos_start"] = s[:, k]
            seg[f"{a}pos_end"] = e[:, k]
        step.run.nseg = n
        L.argot_hip_set_tau_mode(0)
        L.calc_optical_depth_cuda(segp, C.byref(step.cmem), C.byref(step.cpar), C.byref(step.run))
        check("calc_optical_depth_cuda")
        got = np.stack([seg["optical_depth_HI"], seg["optical_depth_HeI"],
                        seg["optical_depth_HeII"]], axis=1).copy()
    finally:
        L.deallocate_pinned_segment(segp)
    want = np.array([P.walk(s[i], e[i])[0] for i in range(n)], np.float32)
    bad = (got.view(np.uint32) != want.view(np.uint32)).any(1)
    assert not bad.any(), (np.flatnonzero(bad)[:5], s[bad][:2], e[bad][:2])
