"""The walk's forms agree bit for bit: the float form of a small mesh, and the
32-bit offset form (taken where the cell sizes leave the float form's
quotients no room) on the same mesh with the box scaled by a power of two,
which scales every length and optical depth exactly.  And the float form's
segments that do not end cleanly in a cell, against the oracle."""
import ctypes as C

import numpy as np
import pytest

from argot_amd import abi, ic
from argot_amd import radiation as R
from argot_amd._lib import check, lib
from helpers import oracle_problem, ragged_workload, small_workload

pytestmark = pytest.mark.gpu

SCALE = 2.0 ** 26    # cells of 2^22 and more: beyond the float form


def scaled(step):
    """The step's box, cells and sources times SCALE, lengths in the unit's
    SCALE-th part."""
    r = step.run
    for a in "xyz":
        setattr(r, f"{a}max", SCALE)
        setattr(r, f"{a}max_local", SCALE)
        setattr(r, f"delta_{a}", getattr(r, f"delta_{a}") * SCALE)
    r.lunit /= SCALE
    for s in step.src:
        s.xpos, s.ypos, s.zpos = s.xpos * SCALE, s.ypos * SCALE, s.zpos * SCALE
    return step


@pytest.mark.parametrize("shape,kahan", [((16, 16, 16), 0), ((12, 10, 14), 0), ((5, 33, 8), 1)])
def test_step_in_a_scaled_box_has_the_same_bits(require_gpu, shape, kahan):
    w = ragged_workload(shape, nsrc=7, seed=71)
    a = R.PointSourceStep(w, tau_mode=kahan)
    sa = a.step()
    ra = a.rates()
    b = scaled(R.PointSourceStep(w, tau_mode=kahan))
    sb = b.step()
    rb = b.rates()
    lib().argot_hip_set_tau_mode(0)
    assert (sa["nray"], sa["ncross"]) == (sb["nray"], sb["ncross"])
    assert sa["nray"] > 0
    assert np.array_equal(ra.view(np.uint32), rb.view(np.uint32))


@pytest.mark.parametrize("shape", [(16, 16, 16), (12, 7, 20)])
def test_segments_ending_on_faces_edges_and_outside(require_gpu, shape):
    w = ragged_workload(shape, nsrc=2, seed=73)
    P = oracle_problem(w)
    step = R.PointSourceStep(w)
    rng = np.random.default_rng(74)
    n = 3000
    size = np.array(shape)
    s = rng.uniform(0.0, 1.0, (n, 3)).astype(np.float32)
    # ends on 0 to 3 cell faces at once, an ulp to either side or exactly there
    e = rng.uniform(0.0, 1.0, (n, 3)).astype(np.float32)
    face = (rng.integers(0, size + 1, (n, 3)) / size).astype(np.float32)
    ulp = rng.integers(-1, 2, (n, 3))
    face = np.where(ulp < 0, np.nextafter(face, np.float32(-1)),
                    np.where(ulp > 0, np.nextafter(face, np.float32(2)), face))
    on = rng.random((n, 3)) < 0.5
    e[on] = face[on]
    e[::10] = rng.uniform(-0.3, 1.3, e[::10].shape)     # and ends outside the box
    s[::17, 1] = e[::17, 1]                              # in a coordinate plane
    s[::19, :2] = e[::19, :2]                            # along an axis
    s[::23] = e[::23]                                    # of no length
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
    assert not bad.any(), (np.flatnonzero(bad)[:5], s[bad][:2], e[bad][:2], got[bad][:2],
                           want[bad][:2])
