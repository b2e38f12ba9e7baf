"""The quadrature rule's limits hold for every ray they admit, whatever part of
its spectrum the other species leave: smooth spectra with a line, a step or
noise added, on columns of HI, HeI and HeII drawn independently, against the
sum over all 256 bins in 64 bits."""
import ctypes as C

import numpy as np
import pytest

from argot_amd import radiation as R
from argot_amd._lib import check, lib
from helpers import cell_centre, oracle_problem, rel_err, small_workload
from test_rate_rule import EDGE, arrays, full_sum, node_sum, rule, tables


def blackbody(nu, t):
    x = 6.626e-27 * 3.28e15 / 1.38066e-16 / t
    v = nu ** 3 / np.expm1(x * nu)
    return v / v.max()


def raised(v, bins, by):
    v = np.array(v, np.float64)
    v[bins] *= by
    return v / v.max()


def spectra(nu):
    rng = np.random.default_rng(11)
    spike = blackbody(nu, 1e5)
    spike[30] += 1.0
    down = nu ** -2.0
    down[44:] *= 0.1
    low = blackbody(nu, 1e5)
    low[44:] = 0.0
    s = {"below the HeI edge": low,
         "5e4 K, one bin up": raised(blackbody(nu, 5e4), 6, 1.3),
         "5e4 K, 38 bins up": raised(blackbody(nu, 5e4), slice(6, 44), 1.3),
         "nu^-6, one bin up": raised(nu ** -6.0, 36, 1.3),
         "1e5 K, one bin up": raised(blackbody(nu, 1e5), 6, 1.3),
         "1e5 K, noise below the HeI edge":
             raised(blackbody(nu, 1e5), slice(0, 44), 1 + 0.05 * rng.standard_normal(44)),
         "1e5 K and a line at 1.5": spike / spike.max(),
         "nu^-2, a step at the HeI edge": down}
    for i in range(60):   # a line, a step or noise of any strength anywhere
        v = blackbody(nu, 10 ** rng.uniform(4.3, 5.7)) if i % 2 else nu ** rng.uniform(-7, 2)
        a, b = sorted(rng.integers(0, 257, 2))
        by = 10 ** rng.uniform(-5, 1)
        if i % 3 == 0:
            v = raised(v, a % 256, 1 + by)
        elif i % 3 == 1:
            v = raised(v, slice(a, b), 1 + by)
        else:
            v = raised(v, slice(0, 256), np.abs(1 + min(by, 0.3) * rng.standard_normal(256)))
        s[f"drawn {i}"] = v / v.max()
    return {k: v.astype(np.float32) for k, v in s.items()}


def columns(rng, sig, n, lam):
    """Columns [n, 3] of independent species whose largest edge optical depth
    (of EDGE) is lam or below."""
    u = 10 ** rng.uniform(-3.0, 0.0, (n, 3))
    for s in range(3):
        u[s::4, s] = 1.0
    u /= sig.max(1)
    k1, k2 = (int(np.argmax(sig[s] > 0)) for s in (1, 2))
    edge = (u @ sig[:, [0, k1, k2]] / EDGE).max(1)
    return u * (lam * rng.random(n) ** 0.3 / edge)[:, None]


def depth_of_sum(sig, hsig, spec, t, d, want):
    """[n, 6]: mean optical depth of the bins, weighted as they enter the sums."""
    tau, y = t @ sig, d @ sig
    f = np.exp(-(tau - tau[:, -1:])) * np.where(y > 1e-12, -np.expm1(-y) / np.maximum(y, 1e-300), 1)
    f = f * spec * (np.abs(tau) + y)
    return np.concatenate([f @ sig.T, f @ hsig.T], 1) / np.where(want > 0, want, 1.0)


def test_rays_within_the_limit_have_the_sum_over_bins():
    run = tables()
    nu, sig, hsig = arrays(run)
    sp = spectra(nu)
    _, qs, qd, w, lim = rule(run, np.array(list(sp.values())))
    qs, qd, w = (a.astype(np.float64) for a in (qs, qd, w))
    rng = np.random.default_rng(5)
    bad = {}
    tried = 0
    for i, (name, s) in enumerate(sp.items()):
        if not lim[i] > 0.0:
            continue
        n = 1500
        far = columns(rng, sig, n, lim[i])
        part = rng.random((n, 1)) ** 2     # the cell's share of the far side's columns
        t, d = far * (1 - part), far * part
        want = full_sum(sig, hsig, s.astype(np.float64), t, d)
        got = node_sum(sig, qs, qd, w[i], t, d)
        nz = want > 0
        # 1e-7 on the test columns, twice that between them, and the FP32
        # rounding of the weights and of the nodes' cross-sections (6e-8 of the
        # optical depths, the cell's included, where the sum comes from)
        depth = depth_of_sum(sig, hsig, s.astype(np.float64), t, d, want)
        tol = 2e-7 + 6e-8 * (1.0 + depth)
        over = np.max(np.abs(got - want)[nz] / want[nz] / tol[nz])
        if not over < 1.0 or np.any(got[~nz]):
            bad[name] = float(over)
        tried += 1
    assert tried > 20
    assert not bad, bad


def limits(cmem, run, spec):
    spec = np.ascontiguousarray(spec, np.float32)
    w, lim = np.zeros((len(spec), 192), np.float32), np.zeros((len(spec), 4), np.float32)
    lib().argot_hip_rate_limits(cmem, C.byref(run), spec.ctypes.data, len(spec), w.ctypes.data,
                                lim.ctypes.data)
    check("argot_hip_rate_limits")
    return w, lim


def test_each_range_holds_to_its_own_limit():
    run = tables()
    nu, sig, hsig = arrays(run)
    sp = spectra(nu)
    rows = np.array(list(sp.values()))
    _, qs, qd, w, lim = rule(run, rows)
    w2, lims = limits(None, run, rows)
    assert np.array_equal(w, w2) and np.array_equal(lim, lims[:, :3].min(1))
    assert (lims[:, 3] >= lims[:, 0]).all()
    # (scales beyond 1.3 are too far apart for the first range's own limit: 3e-7
    # between 1.3 and 1.7 on a spectrum with 1e-7 at both)
    assert (lims[:, 0] <= np.float32(1.3)).all() and (lims[:, 0] == np.float32(1.3)).any()
    # a line below the HeI edge leaves the other ranges their limits
    _, smooth = limits(None, run, (blackbody(nu, 1e5) / blackbody(nu, 1e5)[44:].max())[None])
    assert np.array_equal(lims[list(sp).index("1e5 K, one bin up"), 1:3], smooth[0, 1:3])
    k = [0, *(int(np.argmax(sig[s] > 0)) for s in (1, 2)), 256]
    rng = np.random.default_rng(6)
    node = [slice(0, 12), slice(12, 24), slice(24, 44)]
    tried = np.zeros(3, int)
    for i, s in enumerate(rows.astype(np.float64)):
        for g in range(3):
            if not lims[i, g] > 0.0:
                continue
            tried[g] += 1
            n = 400
            u = 10 ** rng.uniform(-3.0, 0.0, (n, 3)) * (np.arange(3) <= g)
            u /= np.where(np.arange(3) <= g, sig[:, k[g]], 1.0)
            t = u * (EDGE[g] * lims[i, g] * rng.random(n) ** 0.3 / (u @ sig[:, k[g]]))[:, None]
            band = slice(k[g], k[g + 1])
            f = np.exp(-(t @ (sig[:, band] - sig[:, k[g + 1] - 1:k[g + 1]]))) * s[band]
            want = np.concatenate([f @ sig[:, band].T, f @ hsig[:, band].T], 1)
            # the range's nodes; their FP32 differences to the last bin are taken
            # back to those to the range's last bin
            part = (np.arange(44) >= node[g].start) & (np.arange(44) < node[g].stop)
            fn = np.exp(-(t @ (qd + (sig[:, -1:] - sig[:, k[g + 1] - 1:k[g + 1]])))) * part
            rows6 = np.zeros((6, 44))
            o = (0, 24, 72)[g]
            for sp_ in range(g + 1):
                for h in range(2):
                    m = node[g].stop - node[g].start
                    rows6[3 * h + sp_, node[g]] = w[i, o:o + m]
                    o += m
            got = fn @ rows6.T / 2.0 ** 60
            nz = want > 0
            # as above; the differences' rounding: 6e-8 of the range's own depths
            depth = np.concatenate([(f * (t @ sig[:, band])) @ sig[:, band].T,
                                    (f * (t @ sig[:, band])) @ hsig[:, band].T], 1)[nz] / want[nz]
            err = np.abs(got - want)[nz] / want[nz]
            assert (err < 2e-7 + 6e-8 * (1.0 + depth)).all(), (list(sp)[i], g, err.max())
    assert (tried > 20).all(), tried


def test_the_first_ranges_loose_limit():
    """Five times kRuleLoose: what the rays' share of it counts on."""
    run = tables()
    nu, sig, hsig = arrays(run)
    rows = np.array(list(spectra(nu).values()))
    _, qs, qd, w, _ = rule(run, rows)
    _, lims = limits(None, run, rows)
    k1 = int(np.argmax(sig[1] > 0))
    rng = np.random.default_rng(8)
    assert (lims[:, 3] >= 1.7).sum() > 20
    for i, s in enumerate(rows.astype(np.float64)):
        t = EDGE[0] * lims[i, 3] * rng.random((500, 1)) / sig[0, 0]
        f = np.exp(-t * (sig[0, :k1] - sig[0, k1 - 1])) * s[:k1]
        fn = np.exp(-t * (qd[0, :12] + (sig[0, -1] - sig[0, k1 - 1])))
        for h, x in enumerate((sig, hsig)):
            want, got = f @ x[0, :k1], fn @ w[i, 12 * h:12 * h + 12].astype(np.float64) / 2.0 ** 60
            assert (np.abs(got - want) <= 5e-2 * want).all(), (i, h)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 67, 4096 + 5])   # one block, a part of one, wide blocks
def test_device_weights_and_limits_are_the_hosts(require_gpu, n):
    step = R.PointSourceStep(small_workload(n=8, nsrc=1))
    rows = np.array(list(spectra(arrays(step.run)[0]).values()))
    rows[3, 100] = np.nan
    rows[4] = 0.0
    rows = np.resize(rows, (n, 256))
    print(f"rate limits of {n} spectra", flush=True)
    w, lim = limits(C.byref(step.cmem), step.run, rows)
    w0, lim0 = limits(None, step.run, rows)
    assert np.array_equal(lim, lim0)
    assert np.array_equal(w.view(np.uint32), w0.view(np.uint32)) or np.array_equal(
        w[~np.isnan(w)], w0[~np.isnan(w0)])


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["5e4 K, one bin up", "5e4 K, 38 bins up", "nu^-6, one bin up",
                                  "1e5 K, one bin up", "1e5 K, noise below the HeI edge",
                                  "below the HeI edge"])
@pytest.mark.parametrize("cell", [0.05, 30.0])
def test_rates_of_rays_by_ranges_against_the_oracle(require_gpu, name, cell):
    """Single rays through calc_photoion_rate_cuda whose species' columns are
    drawn independently: some ranges within the spectrum's limits, some not."""
    w = small_workload(n=16, nsrc=2, seed=71)
    n = w.n ** 3
    rng = np.random.default_rng(72)
    w.dens = (cell * (0.1 + rng.random(w.dens.shape))).astype(np.float32)
    step, P = R.PointSourceStep(w), oracle_problem(w)
    nu, sig, _ = arrays(step.run)
    spec = spectra(nu)[name]
    row = 1.0e58 * spec.astype(np.float64)
    far = columns(rng, sig, n, 1.0) * np.choose(np.arange(n) % 4, [0.1, 0.5, 1.2, 2.0])[:, None]
    idx = np.stack(np.unravel_index(np.arange(n), w.dens.shape), 1)
    src = rng.uniform(-0.1, 1.1, (n, 3)).astype(np.float32)
    col = w.lunit * w.denstonh
    f = np.stack([w.fHI, w.helium_fact * w.fHeI, w.helium_fact * w.fHeII], 3).reshape(n, 3)
    delta = np.array([P.delta_length(*(float(v) for v in d)) for d in cell_centre(idx, w.n) - src])
    d = w.dens.reshape(n, 1).astype(np.float64) * f * delta[:, None]
    tau = np.maximum(far / col - 0.5 * d, 0.5 * d).astype(np.float32)
    print(f"rates by ranges: {name}, cells {cell}", flush=True)
    got = rates_of(step, src, row, idx, tau)
    want = np.array([P.ray_rate(src[i], row, *(int(v) for v in idx[i]), tau[i], mode=1)
                     for i in range(n)])
    fin = np.isfinite(want) & (want > 1e-30) & (want < 1e37)
    assert fin[:, 0].mean() > 0.4
    # FP32 sums: optical depths of up to about 20 where a sum comes from, rounded
    # to 6e-8 a few times over
    err = rel_err(got[fin], want[fin], 1e-30)
    assert err.max() < 8e-6, err.max()


def rates_of(step, src, row, idx, tau):
    """Rates of one ray to each cell through calc_photoion_rate_cuda."""
    n = len(idx)
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
    return step.rates()


@pytest.mark.gpu
@pytest.mark.parametrize("temp", [3e4, 1e5, 4e5])
@pytest.mark.parametrize("cell", [0.005, 0.3])
def test_node_sums_round_like_fp32(require_gpu, temp, cell):
    """Rays within all limits: the error's root mean square is that of FP32
    rounding (some six roundings of at most 6e-8 on depths of up to 4 where the
    sums come from), with no offset of the forms."""
    w = small_workload(n=16, nsrc=2, seed=81)
    n = w.n ** 3
    rng = np.random.default_rng(82)
    w.dens = (cell * (0.1 + rng.random(w.dens.shape))).astype(np.float32)
    step, P = R.PointSourceStep(w), oracle_problem(w)
    nu, sig, _ = arrays(step.run)
    spec = blackbody(nu, temp).astype(np.float32)
    _, lims = limits(None, step.run, spec[None])
    far = columns(rng, sig, n, 0.9 * lims[0, :3].min())
    idx = np.stack(np.unravel_index(np.arange(n), w.dens.shape), 1)
    src = rng.uniform(-0.1, 1.1, (n, 3)).astype(np.float32)
    tau = (far / (w.lunit * w.denstonh)).astype(np.float32)
    row = 1.0e58 * spec.astype(np.float64)
    print(f"rounding of node sums: {temp:.0e} K, cells {cell}", flush=True)
    got = rates_of(step, src, row, idx, tau)
    want = np.array([P.ray_rate(src[i], row, *(int(v) for v in idx[i]), tau[i], mode=1)
                     for i in range(n)])
    fin = np.isfinite(want) & (want > 1e-30) & (want < 1e37)
    assert fin.all(1).mean() > 0.4
    err = (got[fin] - want[fin]) / want[fin]
    assert np.sqrt(np.mean(err ** 2)) < 2e-7, np.sqrt(np.mean(err ** 2))
