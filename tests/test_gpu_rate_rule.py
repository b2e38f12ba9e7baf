"""Rates of single rays through calc_photoion_rate_cuda on both sides of the
quadrature rule's limits: thin and thick columns, thin and thick cells, one
spectrum with a high limit, a steep one with a lower limit and one with none,
and rays FP32 cannot serve, against the oracle's 64-bit rates."""
import ctypes as C

import numpy as np
import pytest

from argot_amd import abi
from argot_amd import radiation as R
from argot_amd._lib import check, lib
from helpers import cell_centre, oracle_problem, rel_err, small_workload
from test_rate_rule import arrays, columns, spectra, tables

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,limit", [("blackbody 1e+05", 3.0), ("blackbody 3e+04", 1.0),
                                        ("line", 0.0)])
@pytest.mark.parametrize("cell", [0.05, 30.0])
def test_rays_on_both_sides_of_the_limit(require_gpu, name, limit, cell):
    w = small_workload(n=16, nsrc=2, seed=61)
    n = w.n ** 3
    rng = np.random.default_rng(62)
    w.dens = (cell * (0.1 + rng.random(w.dens.shape))).astype(np.float32)
    step, P = R.PointSourceStep(w), oracle_problem(w)
    nu, sig, _ = arrays(tables())
    line = np.zeros(256)
    line[150] = 1.0
    row = 1.0e58 * (line if name == "line" else spectra(nu)[name].astype(np.float64))
    # a quarter each well inside, just inside, just outside and far outside
    scale = (limit or 1.0) * np.choose(np.arange(n) % 4, [0.3, 0.999, 1.001, 1.6])
    far = columns(rng, sig, n, 1.0) * scale[:, None]
    idx = np.stack(np.unravel_index(np.arange(n), w.dens.shape), 1)
    src = rng.uniform(-0.1, 1.1, (n, 3)).astype(np.float32)
    tgt = cell_centre(idx, w.n)
    col = w.lunit * w.denstonh
    f = np.stack([w.fHI, w.helium_fact * w.fHeI, w.helium_fact * w.fHeII], 3).reshape(n, 3)
    delta = np.array([P.delta_length(*(float(v) for v in d)) for d in tgt - src])
    d = w.dens.reshape(n, 1).astype(np.float64) * f * delta[:, None]
    # the column at the far side of the cell is `far`, where the cell leaves room
    tau = np.maximum(far / col - 0.5 * d, 0.5 * d).astype(np.float32)
    # and a few rays no FP32 sum can hold
    src[:3] = tgt[:3]
    rays = R.light_rays(src, np.broadcast_to(row, (n, 256)), idx, tau)
    io = C.c_void_p()
    L = lib()
    L.allocate_pinned_light_ray_IO(C.byref(io), n)
    check("allocate_pinned_light_ray_IO")
    try:
        ctx = (C.byref(step.cmem), C.byref(step.cpar), C.byref(step.run))
        L.zero_out_photoion_rate_cuda(*ctx)
        check("zero_out_photoion_rate_cuda")
        step.run.nray = n
        L.calc_photoion_rate_cuda(ctx[0], rays, io, ctx[1], ctx[2])
        check("calc_photoion_rate_cuda")
    finally:
        L.deallocate_pinned_light_ray_IO(io)
    got = step.rates()
    want = np.array([P.ray_rate(src[i], row, *(int(v) for v in idx[i]), tau[i], mode=1)
                     for i in range(n)])
    # (a rate below FP32's range is compared as zero)
    fin = np.isfinite(want) & (want > 1e-30) & (want < 1e37)
    assert fin[3:].all(1).mean() > 0.4
    # FP32 sums: optical depths of up to about 20 where a sum comes from (the
    # line: up to 30 at its bin), rounded to 6e-8 a few times over
    err = rel_err(got[fin], want[fin], 1e-30)
    assert err.max() < 8e-6, err.max()
    assert np.array_equal(np.isfinite(got[:3]), np.isfinite(want[:3]))
