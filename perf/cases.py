"""The work that a program using this library has it do, as timed cases.

Each case goes through the library's public entry points (the C-ABI of
include/argot_hip.h, by way of argot_amd's host mirror) on inputs made from a
seed.  The kinds:

  step     one point-source pass, step_radiation_tree, on a mesh that stays on
           the GPU: the tree build, every ray's walk, the rates of all cells
  loop     one coupled time step as a hydrodynamics program takes it: the mesh
           sent to the GPU, its chemical time step asked for, then at most five
           passes of transfer, smoothing and chemistry and the update
  chem     the chemistry step alone, on given photoionization rates
  diffuse  one pass of the diffuse (recombination) radiation over all directions
  walk     optical depths of a host list of ray segments
  rates    rates of a host list of rays with known optical depths
  smooth   the 27-point smoothing of the rates on the GPU

exact() gives the outputs in 64 bits from the definitions, in plain torch.
"""
import ctypes as C
import math

import numpy as np
import torch

from argot_amd import abi, ic
from argot_amd import art as A
from argot_amd import radiation as R
from argot_amd._lib import check, lib

THETA = 0.7
YEARS_PER_CODE_TIME = 1.0e8      # ic.TUNIT_S
RATE_COLS = slice(31, 37)        # prev_chem.GammaHI .. HeatHeII in a record of 39 floats


def listed():
    return [
        # The smallest mesh anyone steps (the size of the parity tests and of
        # a smoke test): launches, copies and the tree build are what it costs.
        dict(name="step_16", kind="step", nx=16, ny=16, nz=16, nsrc=6, field="lognormal",
             sources="cells", kahan=False),
        # The comparison-project size: a uniform 64^3 box with a few sources.
        dict(name="step_uniform64", kind="step", nx=64, ny=64, nz=64, nsrc=16, field="uniform",
             sources="cells", kahan=False),
        # A box whose sides are no powers of two and whose cells are not
        # cubes, sources anywhere in their cells.
        dict(name="step_ragged", kind="step", nx=72, ny=58, nz=87, nsrc=250, field="lognormal",
             sources="anywhere", kahan=False),
        # A cosmological box with many galaxies, with the compensated sums
        # that long rays ask for.
        dict(name="step_lognormal128_kahan", kind="step", nx=128, ny=128, nz=128, nsrc=1024,
             field="lognormal", sources="cells", kahan=True),
        # The size the library is quoted on.
        dict(name="step_clumped256", kind="step", nx=256, ny=256, nz=256, nsrc=4096,
             field="lognormal", sources="clumped", kahan=False),
        # A time step of a hydrodynamics run.
        dict(name="loop_64", kind="loop", nx=64, ny=64, nz=64, nsrc=64, field="lognormal",
             sources="anywhere", kahan=False, years=1.0e5),
        # The chemistry of a cosmological box over the same time.
        dict(name="chem_128", kind="chem", nx=128, ny=128, nz=128, nsrc=64, years=1.0e5),
        # The diffuse radiation of a small box, and of the benchmark's box
        # with its 768 directions.
        dict(name="diffuse_32", kind="diffuse", n=32, nside=4),
        dict(name="diffuse_128", kind="diffuse", n=128, nside=8),
        # A host program that keeps its own rays and has their optical depths
        # and rates computed (the reference's call sequence).
        dict(name="walk_list", kind="walk", nx=128, ny=128, nz=128, nseg=1 << 20, kahan=False),
        dict(name="rates_list", kind="rates", nx=64, ny=64, nz=64, nray=1 << 17, nspec=64),
        # The smoothing between transfer and chemistry.
        dict(name="smooth_128", kind="smooth", nx=128, ny=128, nz=128),
    ]


def _log_between(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def _box(rng, lo, hi):
    n = _log_between(rng, lo, hi)
    return {a: max(4, int(n * rng.uniform(0.85, 1.15))) for a in ("nx", "ny", "nz")}


def draw(rng):
    """One more case: every kind, sizes over the logarithm of its range."""
    kind = rng.choice(["step", "step", "step", "step", "loop", "chem", "diffuse", "walk", "rates",
                       "smooth"])
    if kind == "step":
        c = dict(kind=kind, **_box(rng, 16, 144))
        if rng.random() < 0.3:   # a power-of-two cube
            c["nx"] = c["ny"] = c["nz"] = 1 << int(round(math.log2(c["nx"])))
        return dict(c, nsrc=int(_log_between(rng, 1, 1500)),
                    field=rng.choice(["uniform", "lognormal", "lognormal"]),
                    sources=rng.choice(["cells", "anywhere", "clumped"]),
                    kahan=rng.random() < 0.3)
    if kind == "loop":
        return dict(kind=kind, **_box(rng, 16, 64), nsrc=int(_log_between(rng, 2, 64)),
                    field="lognormal", sources="anywhere", kahan=rng.random() < 0.3,
                    years=_log_between(rng, 3.0e4, 2.0e5))
    if kind == "chem":
        return dict(kind=kind, **_box(rng, 24, 110), nsrc=int(_log_between(rng, 2, 64)),
                    years=_log_between(rng, 1.0e4, 2.0e5))
    if kind == "diffuse":
        return dict(kind=kind, n=2 * int(_log_between(rng, 8, 60)), nside=rng.choice([2, 4, 8]))
    if kind == "walk":
        return dict(kind=kind, **_box(rng, 32, 144), nseg=int(_log_between(rng, 1 << 10, 1 << 20)),
                    kahan=rng.random() < 0.3)
    if kind == "rates":
        return dict(kind=kind, **_box(rng, 16, 80), nray=int(_log_between(rng, 1 << 10, 1 << 17)),
                    nspec=int(_log_between(rng, 1, 256)))
    return dict(kind=kind, **_box(rng, 16, 160))


# ------------------------------------------------------------------ inputs ---

def _gen(seed, salt=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * int(seed) + salt)
    return g


def _shape(case):
    return (case["nx"], case["ny"], case["nz"]) if "nx" in case else (case["n"],) * 3


def _uniform(g, shape, lo, hi):
    return torch.rand(shape, generator=g, device="cuda", dtype=torch.float32) * (hi - lo) + lo


def _lognormal(g, shape):
    """exp of a Gaussian field with P(k) ~ k^-3 and unit variance, mean 1."""
    white = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
    k2 = sum(f * f for f in torch.meshgrid(
        *[(torch.fft.fftfreq if d < 2 else torch.fft.rfftfreq)(m, d=1.0 / m, device="cuda")
          for d, m in enumerate(shape)], indexing="ij"))
    k2[0, 0, 0] = 1.0
    amp = k2 ** -0.75
    amp[0, 0, 0] = 0.0
    f = torch.fft.irfftn(torch.fft.rfftn(white) * amp, s=shape)
    f = (f - f.mean()) / f.std()
    return torch.exp(f - 0.5)


def _fields(case, seed):
    """dens, fHI, fHII, fHeI, fHeII, fHeIII on the GPU (FP32)."""
    shape, g = _shape(case), _gen(seed)
    if case["kind"] == "diffuse":
        dens = _lognormal(g, shape)
        x, a, b = (_uniform(g, shape, 0.0, 1.0) for _ in range(3))
        return dens, 1 - x, x, 1 - a, a * (1 - b), a * b
    if case.get("field") == "uniform":
        # one neutral fraction for the whole box, the box's own
        one = torch.ones(shape, device="cuda")
        x = 1.0e-3 * (1.0 + float(torch.rand(1, generator=g, device="cuda")))
        return one, one * (1 - x), one * x, one * (1 - x), one * x, one * 0
    dens = _lognormal(g, shape)
    fHI = _uniform(g, shape, 1.0e-4, 1.0)
    fHeI = _uniform(g, shape, 1.0e-4, 1.0)
    return dens, fHI, 1 - fHI, fHeI, 1 - fHeI, 0 * fHI


def _sources(case, seed):
    """Positions [n, 3] (FP32), photon rates [n] and spectra [n, 256]."""
    shape, n = np.array(_shape(case)), case["nsrc"]
    rng = np.random.default_rng([int(seed), 1])
    how = case.get("sources", "anywhere")
    if how == "clumped":
        centres = rng.uniform(0, 1, (8, 3)) * shape
        p = centres[rng.integers(0, 8, n)] + rng.normal(0.0, 1.0 / 32, (n, 3)) * shape
        pos = (np.clip(np.floor(p), 0, shape - 1) + 0.5) / shape
    elif how == "cells":
        pos = (np.floor(rng.uniform(0, 1, (n, 3)) * shape) + 0.5) / shape
    else:
        pos = rng.uniform(0.02, 0.98, (n, 3))
    if case.get("field") == "uniform":
        rates = np.full(n, 5.0e48)
    else:
        rates = ic.power_law_rates(rng, n)
    # sources at cell centres: 1e5 K, as in the benchmark (their own cells' rates
    # are infinite); elsewhere some cooler ones among them
    cool = (rng.random(n) < 0.2) & (how == "anywhere")
    temps = np.where(cool, 3.0e4, 1.0e5)
    rows = {t: _blackbody(t) for t in (1.0e5, 3.0e4)}
    return pos.astype(np.float32), rates, np.array([rows[t] * q for t, q in zip(temps, rates)])


NBIN, LOG_NU_MAX = abi.NGRID_NU, 1.5


def _blackbody(temp):
    """Photons per bin of a blackbody on the 256 logarithmic bins from the
    Lyman limit to 10^1.5 of it, in sum 1."""
    x, w = np.polynomial.legendre.leggauss(16)
    edge = LOG_NU_MAX * np.arange(NBIN + 1) / NBIN
    mid, half = 0.5 * (edge[1:] + edge[:-1]), 0.5 * (edge[1] - edge[0])
    nu = 10.0 ** (mid[:, None] + half * x)
    y = 6.626e-27 * 3.28e15 / (1.38066e-16 * temp) * nu
    f = (w * nu ** 3 / np.expm1(y)).sum(1)
    return f / f.sum()


def _records(case, seed, rates=None):
    """struct fluid_mesh records [ncell, 39] (FP32) on the GPU."""
    dens, *frac = (f.reshape(-1) for f in _fields(case, seed))
    hfact = ic.helium_fact(0.24)
    rec = torch.zeros((dens.numel(), 39), device="cuda")
    rec[:, 0] = dens
    felec = frac[1] + hfact * (frac[3] + 2.0 * frac[4])
    wmol = 1.0 / ((1.0 + felec.double()) * ic.XHYDROGEN + 0.25 * ic.YHELIUM)
    u = (1.0e4 / (ic.chem_units()["uenetok"] * wmol)).float()
    rec[:, 5] = u
    rec[:, 37] = u
    for at in (11, 24):
        rec[:, at] = wmol.float()
        for k, f in enumerate([felec, *frac]):
            rec[:, at + 1 + k] = f
        if rates is not None:
            rec[:, at + 7:at + 13] = rates
    return rec


def _given_rates(case, seed):
    """Rates [ncell, 6] of the shape a transfer pass leaves: inverse square
    around the sources, cut off exponentially."""
    shape = _shape(case)
    pos, rates, _ = _sources(dict(case, nsrc=case.get("nsrc", 16)), seed)
    axes = [(torch.arange(m, device="cuda") + 0.5) / m for m in shape]
    g = torch.zeros(shape, device="cuda", dtype=torch.float64)
    for p, q in zip(pos, rates):
        r2 = sum((a - float(c)).square().reshape([-1 if k == d else 1 for k in range(3)])
                 for d, (a, c) in enumerate(zip(axes, p))) + 1.0e-4
        g += 1.2e-18 * q / (4 * math.pi * ic.LUNIT_CM ** 2) / r2 * torch.exp(-12.0 * r2.sqrt())
    g = g.reshape(-1, 1) * torch.tensor([1.0, 1.6e-11, 0.9, 0.08, 2.0e-11, 4.0e-12],
                                        device="cuda", dtype=torch.float64)
    return g.float()


class _DeviceMesh:
    """The context's device mesh as an array that keeps its context alive."""

    def __init__(self, step, ncell):
        self.step = step
        self.__cuda_array_interface__ = {
            "shape": (ncell, 39), "typestr": "<f4", "version": 2, "strides": None,
            "data": (int(step.cmem.mesh_dev), False)}


def _device_mesh(step, ncell):
    return torch.as_tensor(_DeviceMesh(step, ncell), device="cuda")


class _Pinned:
    """Pinned host memory from the library's allocators, as an array."""

    def __init__(self, alloc, free, nbytes_each, count):
        self.p, self.free = C.c_void_p(), free
        getattr(lib(), alloc)(C.byref(self.p), count)
        check(alloc)
        self.__array_interface__ = {"shape": (count, nbytes_each), "typestr": "|u1", "version": 3,
                                    "data": (self.p.value, False)}

    def __del__(self):
        try:
            getattr(lib(), self.free)(self.p)
        except Exception:
            pass


class _Diffuse(A.DiffuseStep):
    """A DiffuseStep that gives back its own mesh; the tracing buffers are
    shared by the process."""

    def __del__(self):
        try:
            lib().free_hd_param(C.byref(self.hd))
            lib().argot_hip_release_gpu(C.byref(self.cmem))
        except Exception:
            pass


def _tau_mode(case):
    return 1 if case.get("kahan") else 0


def _context(case, seed, rates=None):
    """A PointSourceStep over the case's mesh and sources, its device mesh
    sent, and the sources' arrays."""
    shape = _shape(case)
    ncell = int(np.prod(shape))
    nsrc = case.get("nsrc", 0) if case["kind"] in ("step", "loop") else 0
    src = (abi.RadiationSrc * max(nsrc, 1))()
    if nsrc:
        pos, _, spec = _sources(case, seed)
        for i in range(nsrc):
            s = src[i]
            s.type, s.param = 0, 1.0e5
            s.xpos, s.ypos, s.zpos = (float(v) for v in pos[i])
            np.ctypeslib.as_array(s.photon_rate)[:] = spec[i]
    freq, cs = R.freq_and_csect()

    class Box:   # what run_param_for reads of a workload
        dens = np.broadcast_to(np.float32(1.0), shape)
        lunit, denstonh = ic.LUNIT_CM, ic.DENSTONH
    Box.nsrc = nsrc
    run = R.run_param_for(Box, freq, cs)
    mesh = abi.mesh_array(ncell)
    host = torch.from_numpy(np.frombuffer(mesh, dtype=np.float32).reshape(ncell, 39))
    host.copy_(_records(case, seed, rates))
    return R.PointSourceStep.from_state(mesh, src, run, ic.helium_fact(0.24),
                                        tau_mode=_tau_mode(case))


def _segments(case, seed):
    """Starts and ends [nseg, 3] (FP32): sixteen sources per target, targets
    in mesh order from a random cell on."""
    shape, n = np.array(_shape(case)), case["nseg"]
    rng = np.random.default_rng([int(seed), 2])
    pool = rng.uniform(0.02, 0.98, (64, 3)).astype(np.float32)
    cell = (rng.integers(0, shape.prod()) + np.arange(n) // 16) % shape.prod()
    idx = np.stack([cell // (shape[1] * shape[2]), cell // shape[2] % shape[1], cell % shape[2]], 1)
    start = pool[(rng.integers(0, 64) + np.arange(n) % 16 * 3) % 64]
    return start, ((idx + 0.5) / shape).astype(np.float32)


def _rays(case, seed):
    """Rays of a host list: source positions, spectra (table, index), target
    cells and optical depths; eight rays to a target."""
    shape, n = np.array(_shape(case)), case["nray"]
    rng = np.random.default_rng([int(seed), 3])
    pool = rng.uniform(0.0, 1.0, (case["nspec"], 3)).astype(np.float32)
    rates = ic.power_law_rates(rng, case["nspec"])
    table = np.array([_blackbody(1.0e5) * q for q in rates])
    ntarget = -(-n // 8)
    first = rng.integers(0, shape.prod())
    cell = (first + np.repeat(np.arange(ntarget), 8)[:n]) % shape.prod()
    # a target met twice when the list is longer than the mesh keeps its rays together
    cell = np.sort(cell)
    idx = np.stack([cell // (shape[1] * shape[2]), cell // shape[2] % shape[1], cell % shape[2]], 1)
    which = (rng.integers(0, case["nspec"], ntarget).repeat(8)[:n] + np.arange(n) % 8) % case["nspec"]
    # columns of neutral gas on the way, in code units: mean density times a path
    path = np.linalg.norm(pool[which] - (idx + 0.5) / shape, axis=1)
    tau = path[:, None] * rng.lognormal(-1.0, 1.0, (n, 3)) * np.array([1.0, 0.08, 0.08])
    return pool[which], (table, which), idx, tau.astype(np.float32)


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.kind, s.case = case["kind"], case
    ncell = int(np.prod(_shape(case)))
    if s.kind == "diffuse":
        f = [v.cpu().numpy() for v in _fields(case, seed)]
        w = ic.Workload("diffuse", case["n"], *f, np.zeros((0, 3), np.float32), np.zeros(0),
                        np.zeros(0, np.float32))
        s.step = _Diffuse(w, nside=case["nside"])
        s.mesh = _device_mesh(s.step, ncell)
        return s
    rates = _given_rates(case, seed) if s.kind in ("chem", "smooth") else None
    s.step = _context(case, seed, rates)
    s.mesh = _device_mesh(s.step, ncell)
    if "years" in case:
        s.dtime = case["years"] / YEARS_PER_CODE_TIME
    if s.kind == "walk":
        n = case["nseg"]
        s.seg = _Pinned("allocate_pinned_segment", "deallocate_pinned_segment", 56, n)
        a = np.asarray(s.seg).view(np.float32)
        a[:] = 0.0
        np.asarray(s.seg).view(np.uint64)[:, 0] = np.arange(n)
        a[:, 4:7], a[:, 7:10] = _segments(case, seed)
        s.tau = a[:, 10:13]
        s.step.run.nseg = n
    elif s.kind == "rates":
        n = case["nray"]
        s.rays = R.light_rays(*_rays(case, seed))
        s.io = _Pinned("allocate_pinned_light_ray_IO", "deallocate_pinned_light_ray_IO",
                       C.sizeof(abi.LightRayIO), n)
        s.step.run.nray = n
    return s


def run(s):
    p, L = s.step, lib()
    ctx = lambda: (C.byref(p.cmem), C.byref(p.cpar), C.byref(p.run))  # noqa: E731
    if s.kind == "step":
        p.step()
        return s.mesh[:, RATE_COLS]
    if s.kind == "loop":
        p.send_mesh()
        dt, _ = p.chem_timestep()
        p.step(dtime=s.dtime, iterations=5)
        return {"dt": dt, "state": s.mesh[:, 24:38], "energy": s.mesh[:, 1]}
    if s.kind == "chem":
        diff = p.chemistry(s.dtime)
        return {"diff": list(diff), "chem": s.mesh[:, 11:24], "uene": s.mesh[:, 5]}
    if s.kind == "diffuse":
        p.step()
        return s.mesh[:, RATE_COLS]
    if s.kind == "walk":
        L.argot_hip_set_helium_fact(p.w.helium_fact)
        L.argot_hip_set_tau_mode(p.tau_mode)
        L.calc_optical_depth_cuda(s.seg.p, *ctx())
        check("calc_optical_depth_cuda")
        return s.tau
    if s.kind == "rates":
        L.argot_hip_set_helium_fact(p.w.helium_fact)
        L.zero_out_photoion_rate_cuda(*ctx())
        check("zero_out_photoion_rate_cuda")
        L.calc_photoion_rate_cuda(C.byref(p.cmem), s.rays, s.io.p, C.byref(p.cpar), C.byref(p.run))
        check("calc_photoion_rate_cuda")
        return s.mesh[:, RATE_COLS]
    L.smooth_photoion_rate(None, C.byref(p.run), C.byref(p.cmem), C.byref(p.cpar), None)
    check("smooth_photoion_rate")
    return s.mesh[:, RATE_COLS]


# -------------------------------------------------------------------- work ---

def _rays_per_cell(case):
    """About how many rays a target gets at theta = 0.7: every source, or
    for many of them some levels of the tree (measured on the listed cases)."""
    n = case["nsrc"]
    if case["sources"] == "clumped":
        return min(n, 29.0)
    return n if n <= 16 else min(n, 16 + 14 * math.log2(n / 16))


def work(case):
    """Bytes: each input read and each output written once.  Operations: a
    crossing costs 3 divisions, 3 sums, the face choice and 3 products
    (about 20), a ray's rates 256 bins of 3 optical depths, 3 weights, the two
    exponentials and 6 sums (about 30), a chemistry sub-step some 3000."""
    shape = _shape(case)
    n = float(np.prod(shape))
    side = n ** (1.0 / 3.0)
    kind = case["kind"]
    if kind in ("step", "loop"):
        rays = n * _rays_per_cell(case)
        w = {"bytes": 40 * n + 2072 * case["nsrc"], "flops": rays * (256 * 30 + 20 * 0.6 * side)}
        if kind == "loop":
            w["bytes"] += 3 * 156 * n
            w["flops"] = 2 * w["flops"] + 3000 * 40 * n * case["years"] / 1.0e5
        return w
    if kind == "chem":
        return {"bytes": 2.0 * 104 * n, "flops": 3000 * 40 * n * case["years"] / 1.0e5}
    if kind == "diffuse":
        return {"bytes": 60 * n, "flops": 12.0 * case["nside"] ** 2 * n * 1.86 * 60}
    if kind == "walk":
        return {"bytes": 16 * n + 36.0 * case["nseg"], "flops": 20.0 * side * case["nseg"]}
    if kind == "rates":
        return {"bytes": 2400.0 * case["nray"] + 40 * n, "flops": 256.0 * 30 * case["nray"]}
    return {"bytes": 48 * n, "flops": 6 * 28 * n}


# ------------------------------------------------------------------- exact ---
# The definitions in 64 bits, in plain torch and numpy.

F64 = dict(device="cuda", dtype=torch.float64)


def _cross_sections():
    """sigma [3, 256] as the tables hold them (rounded to FP32) and the bins'
    frequencies in Lyman limits."""
    nu = 10.0 ** (LOG_NU_MAX * (np.arange(NBIN) + 0.5) / NBIN)

    def hydrogenic(x, pre):
        e = np.sqrt(x - 1.0)
        return pre / x ** 4 * np.exp(4.0 - 4.0 * np.arctan(e) / e) / (1.0 - np.exp(-2 * np.pi / e))

    s = np.zeros((3, NBIN))
    s[0] = hydrogenic(nu, 6.3e-18)
    m = nu >= 1.8125
    s[1][m] = 7.83e-18 * (1.66 * (nu[m] / 1.8125) ** -2.05 - 0.66 * (nu[m] / 1.8125) ** -3.05)
    m = nu >= 4.0
    s[2][m] = hydrogenic(nu[m] / 4.0, 6.3e-18 / 4.0)
    return (torch.tensor(s.astype(np.float32).astype(np.float64), **F64),
            torch.tensor(nu.astype(np.float32).astype(np.float64), **F64))


def _densities(case, seed):
    """nHI, nHeI, nHeII [ncell, 3] in code units and dens."""
    f = [v.reshape(-1).double() for v in _fields(case, seed)]
    h = ic.helium_fact(0.24)
    return torch.stack([f[0] * f[1], f[0] * h * f[3], f[0] * h * f[4]], 1)


def _columns(n3, shape, start, end):
    """Optical depths [n, 3] from start to end [n, 3] through the cells."""
    d = torch.tensor(shape, **F64)
    step, pos = end - start, start.clone()
    length = step.square().sum(1).sqrt()
    cell = (pos * d).floor().long()
    last = (end * d).floor().long()
    lim = torch.tensor(shape, device="cuda") - 1
    cell = torch.minimum(cell.clamp(min=0), lim)
    last = torch.minimum(last.clamp(min=0), lim)
    up = (step > 0).long()
    sign = 2 * up - 1
    inv = torch.where(step == 0, torch.full_like(step, 1e300), 1.0 / step)
    at = torch.zeros(len(start), **F64)   # place on the line, 0 to 1
    tau = torch.zeros(len(start), 3, **F64)
    stride = torch.tensor([shape[1] * shape[2], shape[2], 1], device="cuda")
    for _ in range(int(sum(shape)) + 3):
        going = (cell != last).any(1)
        t = torch.where(step == 0, torch.full_like(step, 1e300), ((cell + up) / d - start) * inv)
        # an axis that has come to its last cell crosses no more faces
        t = torch.where(cell == last, torch.full_like(t, 1e300), t)
        nxt, ax = t.min(1)
        nxt = torch.where(going, nxt.clamp(max=1.0), torch.ones_like(nxt))
        nxt = torch.maximum(nxt, at)
        tau += ((nxt - at) * length)[:, None] * n3[(cell * stride).sum(1)]
        at = nxt
        if not bool(going.any()):
            break
        move = torch.nn.functional.one_hot(ax, 3) * going[:, None].long()
        cell = cell + move * sign
    return tau


def _ray_rates(case, n3, cell, src, tau, spec, row, sig, nu):
    """Rates [n, 6] of rays with spectra spec[row] and columns tau to the
    centres of the target cells."""
    shape = _shape(case)
    tiny, lu = 1.0e-31, ic.LUNIT_CM
    hfact_n = n3[cell] * ic.DENSTONH
    idx = torch.stack([cell // (shape[1] * shape[2]), cell // shape[2] % shape[1],
                       cell % shape[2]], 1)
    size = 1.0 / torch.tensor(shape, **F64)
    d = (idx + 0.5) * size - src
    r2 = d.square().sum(1)
    dl = (r2 + tiny).sqrt()
    dxy = (d[:, :2].square().sum(1) + tiny).sqrt()
    cosines = torch.stack([d[:, 0] / dxy * (dxy / dl), d[:, 1] / dxy * (dxy / dl), d[:, 2] / dl], 1)
    delta = (size / cosines.abs().clamp(min=tiny)).min(1).values
    dist = r2.sqrt()
    dtau = hfact_n * (delta * lu)[:, None]
    col = tau * (lu * ic.DENSTONH) - 0.5 * dtau
    vol = 4 * math.pi / 3 * ((dist + 0.5 * delta) ** 3 - (dist - 0.5 * delta) ** 3) * lu ** 3
    r = 1.0 / (hfact_n * vol[:, None] + tiny)
    out = torch.empty(len(cell), 6, **F64)
    edge = (1.0, 1.8125, 4.0)
    for a in range(0, len(cell), 1 << 18):
        b = slice(a, a + (1 << 18))
        w = dtau[b, :, None] * sig
        dtot = w.sum(1)
        depth = (col[b, :, None] * sig).sum(1)
        absorbed = spec[row[b]] * torch.exp(-depth) * -torch.expm1(-dtot)
        for k in range(3):
            g = w[:, k] / (dtot + tiny) * absorbed * r[b, k, None]
            out[b, (0, 2, 3)[k]] = g.sum(1)
            h = torch.where(nu > edge[k], g * (nu - edge[k]), torch.zeros_like(g))
            out[b, (1, 4, 5)[k]] = h.sum(1) * (6.626e-27 * 3.28e15)
    return out


class _Node:
    pass


def _tree(pos, spec):
    """The source oct-tree: nodes with centre, squared length, spectrum and
    children; key digits as the box is halved."""
    key = (pos.astype(np.float32).astype(np.float64) * (1 << 21)).astype(np.int64)
    lum = spec.sum(1)

    def node(members, level, weight):
        t = _Node()
        t.n, t.level = len(members), level
        t.len2 = 4.0 ** -level
        w = weight[members]
        t.centre = (pos[members].astype(np.float64) * w[:, None]).sum(0) / w.sum()
        t.spec, t.kids, t.members = spec[members].sum(0), [], members
        if (len(members) > 1 or level == 0) and level < 21:
            b = (key[members] >> (20 - level)) & 1
            octant = (b[:, 0] << 2) | (b[:, 1] << 1) | b[:, 2]
            t.kids = [node(members[octant == o], level + 1, lum) for o in range(8)
                      if (octant == o).any()]
        return t

    return node(np.arange(len(pos)), 0, spec[:, 0])


def _exact_step(case, seed):
    shape = _shape(case)
    ncell = int(np.prod(shape))
    n3 = _densities(case, seed)
    pos, _, spec = _sources(case, seed)
    size = 1.0 / torch.tensor(shape, **F64)
    every = torch.arange(ncell, device="cuda")

    def centre(c):
        i = torch.stack([c // (shape[1] * shape[2]), c // shape[2] % shape[1], c % shape[2]], 1)
        return (i + 0.5) * size

    target = centre(every)
    cells, srcs, rows, spectra = [], [], [], []

    def emit(c, p, s):
        cells.append(c)
        srcs.append(torch.tensor(p, **F64).expand(len(c), 3))
        rows.append(torch.full((len(c),), len(spectra), device="cuda"))
        spectra.append(s)

    def visit(t, c):
        r2 = (target[c] - torch.tensor(t.centre, **F64)).square().sum(1)
        far = r2 * (THETA * THETA) > t.len2
        if bool(far.any()):
            emit(c[far], t.centre, t.spec)
        c = c[~far]
        if not len(c):
            return
        if t.n > 1:
            for k in t.kids:
                visit(k, c)
        else:
            emit(c, pos[t.members[0]].astype(np.float64), spec[t.members[0]])

    visit(_tree(pos, spec), every)
    cells, srcs, rows = torch.cat(cells), torch.cat(srcs), torch.cat(rows)
    spectra = torch.tensor(np.array(spectra), **F64)
    sig, nu = _cross_sections()
    total = torch.zeros(ncell, 6, **F64)
    for a in range(0, len(cells), 1 << 21):
        b = slice(a, a + (1 << 21))
        tau = _columns(n3, shape, srcs[b], target[cells[b]])
        g = _ray_rates(case, n3, cells[b], srcs[b], tau, spectra, rows[b], sig, nu)
        total.index_add_(0, cells[b], g)
    return total


def _exact_smooth(case, seed):
    shape = _shape(case)
    v = _given_rates(case, seed).double().reshape(*shape, 6).permute(3, 0, 1, 2)
    p = torch.nn.functional.pad(v[None], (1,) * 6, mode="replicate")[0]
    s = 29.0 * v
    for i in range(3):
        for j in range(3):
            for k in range(3):
                s = s + p[:, i:i + shape[0], j:j + shape[1], k:k + shape[2]]
    return (s / 56.0).permute(1, 2, 3, 0).reshape(-1, 6)


def _directions(nside):
    """HEALPix ring centres: unit vectors and the entry face (0 to 5: up and
    down z, x, y) each direction's rays start on."""
    npix, ncap = 12 * nside * nside, 2 * nside * (nside - 1)
    out, face = [], []
    for p in range(npix):
        if p < ncap:
            i = int((1 + math.isqrt(1 + 2 * p)) // 2)
            j = p + 1 - 2 * i * (i - 1)
            z, phi = 1.0 - i * i * (4.0 / npix), (j - 0.5) * (0.5 * math.pi) / i
        elif p < npix - ncap:
            q = p - ncap
            i, j = q // (4 * nside) + nside, q % (4 * nside) + 1
            off = 1.0 if (i + nside) & 1 else 0.5
            z, phi = (2 * nside - i) * (2.0 / (3.0 * nside)), (j - off) * math.pi / (2 * nside)
        else:
            q = npix - p
            i = int((1 + math.isqrt(2 * q - 1)) // 2)
            j = 4 * i + 1 - (q - 2 * i * (i - 1))
            z, phi = -1.0 + i * i * (4.0 / npix), (j - 0.5) * (0.5 * math.pi) / i
        th = math.acos(z)
        ct, st, cp, sp, tt = math.cos(th), math.sin(th), math.cos(phi), math.sin(phi), math.tan(th)
        out.append([c if abs(c) > 1e-31 else (1e-31 if c >= 0 else -1e-31)
                    for c in (st * cp, st * sp, ct)])
        a, b = (cp, 2) if abs(cp) >= math.cos(math.pi / 4) else (sp, 4)
        lim = 1.0 / abs(a)
        face.append(0 if 0 <= tt <= lim else 1 if -lim <= tt < 0 else b if a >= 0 else b + 1)
    return np.array(out, np.float32).astype(np.float64), np.array(face)


def _medium(case, seed):
    """Absorption coefficients and source functions [ncell, 3] of the three
    bands."""
    dens, fHI, fHII, fHeI, fHeII, fHeIII = (v.reshape(-1).double() for v in _fields(case, seed))
    h, nH = ic.helium_fact(0.24), dens * ic.DENSTONH
    nHI, nHII = fHI * nH, fHII * nH
    nHeI, nHeII, nHeIII = fHeI * h * nH, fHeII * h * nH, fHeIII * h * nH
    ne = nHII + nHeII + 2 * nHeIII
    t = 1.0e4
    lam = [2.0 * e / t for e in (157807.0, 285335.0, 631515.0)]
    tev = t * 8.61623e-5
    lt = math.log(tev)
    a2 = math.exp(sum(c * lt ** k for k, c in enumerate((
        -28.61303380689232, -0.7241125657826851, -0.02026044731984691, -0.002380861877349834,
        -0.0003212605213188796, -0.00001421502914054107, 4.989108920299513e-6,
        5.755614137575758e-7, -1.856767039775261e-8, -3.071135243196595e-9))))
    b2 = 2.753e-14 * lam[0] ** 1.5 / (1 + (lam[0] / 2.740) ** 0.407) ** 2.242
    a4 = 3.92e-13 / tev ** 0.6353
    if tev > 0.8:
        a4 += 1.54e-9 * (1 + 0.3 / math.exp(8.099328789667 / tev)) / (
            math.exp(40.49664394833662 / tev) * tev ** 1.5)
    b4 = 1.26e-14 * lam[1] ** 0.75
    a6 = 3.36e-10 / math.sqrt(t) / (t / 1.e3) ** 0.2 / (1.0 + (t / 1.e6) ** 0.7)
    b6 = 1.3765e-14 * lam[2] ** 1.5 / (1 + (lam[2] / 2.740) ** 0.407) ** 2.242
    aHI, aHeI, aHeII = (f(e) * n for (f, e), n in zip(_EDGES, (nHI, nHeI, nHeII)))
    k = torch.stack([aHI + 1e-31, aHI * 1.9529766579e-01 + aHeI + 1e-31,
                     aHI * 1.9513732355e-02 + aHeI * 2.6858709594e-01 + aHeII + 1e-31], 1)
    ev = 13.6 * 1.6022e-12 / (4 * math.pi)
    s = torch.stack([(a2 - b2) * ne * nHII * ev, (a4 - b4) * ne * nHeII * ev * 1.8125,
                     (a6 - b6) * ne * nHeIII * ev * 4.0], 1) / k
    return k, s


def _hydrogenic(nu, edge, pre):
    e = math.sqrt(nu / edge - 1.0)
    return pre * (edge / nu) ** 4 * math.exp(4 - 4 * math.atan(e) / e) / (1 - math.exp(-2 * math.pi / e))


_EDGES = ((lambda nu: _hydrogenic(nu, 1.0, 6.3e-18), 1.0 + 1e-7),
          (lambda nu: 7.83e-18 * (1.66 * (nu / 1.8125) ** -2.05 - 0.66 * (nu / 1.8125) ** -3.05),
           1.8125 + 1e-7),
          (lambda nu: _hydrogenic(nu, 4.0, 6.3e-18 / 4.0), 4.0 + 1e-7))


def _band_factors():
    """Photoionization and heating per mean intensity of the three bands: the
    reference's sums over 64 intervals above each edge."""
    out = []
    for (cs, _), unit, nu_l in zip(_EDGES, (1.0, 1.8125, 4.0), (3.2885e15, 5.9483e15, 1.3154e16)):
        w, g0, g1 = 0.0632353 / 64, 0.0, 0.0
        for i in range(64):
            a, b = unit + i * w + (1e-7 if i == 0 else 0.0), unit + (i + 1) * w
            ca, cb = (4 * math.pi * cs(v) / (6.626e-27 * (v * nu_l)) for v in (a, b))
            g0 += 0.5 * (ca + cb)
            g1 += 0.5 * ((0.0 if i == 0 else ca * (a - unit)) + ca * (b - unit))
        out.append((g0 / 64, g1 / (64 / (6.626e-27 * nu_l))))
    return out


def _exact_diffuse(case, seed):
    n = case["n"]
    kap, src = _medium(case, seed)
    ovr, face = _directions(case["nside"])
    half, ncell, h = n // 2, n ** 3, 1.0 / n
    off = torch.tensor([0.521212345, 0.508512345, 0.468287655], **F64)
    stride = torch.tensor([n * n, n, 1], device="cuda")
    total = torch.zeros(ncell, 6, **F64)
    per = max(1, (3 << 30) // (ncell * 4 * 8))
    rj = (1.128855608262e-01, 5.288790581895e-03, 1.2404369898e-01)
    rh = (3.1154224364e+00, 5.2452188546e-01, 8.7872474963e+00)
    f = _band_factors()
    a, b = torch.meshgrid(torch.arange(half, device="cuda"), torch.arange(half, device="cuda"),
                          indexing="ij")
    for d0 in range(0, len(ovr), per):
        dirs = torch.tensor(ovr[d0:d0 + per], **F64)
        fc = torch.tensor(face[d0:d0 + per], device="cuda")
        nd = len(dirs)
        acc = torch.zeros(nd * ncell, 4, **F64)
        dom = torch.tensor([2, 2, 0, 0, 1, 1], device="cuda")[fc]
        others = torch.tensor([[0, 1], [1, 2], [0, 2]], device="cuda")[torch.tensor(
            [0, 0, 1, 1, 2, 2], device="cuda")[fc]]
        for group in range(4):
            u, v = (2 * a + (group >> 1)).reshape(-1), (2 * b + (group & 1)).reshape(-1)
            start = torch.zeros(nd, half * half, 3, dtype=torch.long, device="cuda")
            start.scatter_(2, others[:, None, :1].expand(nd, half * half, 1), u[None, :, None]
                           .expand(nd, -1, 1))
            start.scatter_(2, others[:, None, 1:].expand(nd, half * half, 1), v[None, :, None]
                           .expand(nd, -1, 1))
            x = (start + off) * h
            entry = (fc & 1).double()
            x.scatter_(2, dom[:, None, None].expand(nd, half * half, 1),
                       entry[:, None, None].expand(nd, half * half, 1))
            o = dirs[:, None].expand_as(x).reshape(-1, 3)
            x = x.reshape(-1, 3)
            cell = (x * n).floor().long()
            cell = torch.where((o < 0) & (cell == n), cell - 1, cell)
            m = dom[:, None].expand(nd, half * half).reshape(-1, 1)
            base = (torch.arange(nd, device="cuda") * ncell)[:, None].expand(
                nd, half * half).reshape(-1)
            up = (o > 0).long()
            I = torch.zeros(len(x), 3, **F64)
            while len(x):
                r = (((cell + up) * h - x) / o).clamp(min=0.0)
                rmin = r.min(1, keepdim=True).values
                here = (cell * stride).sum(1)
                k, s = kap[here], src[here]
                dl = rmin * ic.LUNIT_CM
                e1 = -torch.expm1(-k * dl)
                acc[base + here] += torch.cat([dl, I * e1], 1)
                I = I * (1 - e1) + s * e1
                x = x + rmin * o
                cell = cell + torch.where(r == rmin, 2 * up - 1, torch.zeros_like(up))
                gone = (cell < 0) | (cell >= n)
                end = gone.gather(1, m)[:, 0]
                side = gone.any(1) & ~end
                x = torch.where(gone, (cell < 0).double(), x)
                cell = torch.where(gone, cell % n, cell)
                I = torch.where(side[:, None], torch.zeros_like(I), I)
                keep = ~end
                x, cell, o, m, base, up, I = (q[keep] for q in (x, cell, o, m, base, up, I))
        acc = acc.reshape(nd, ncell, 4)
        for d in range(nd):
            q = acc[d, :, 1:] / kap / acc[d, :, :1] + src
            for c, terms in ((0, (1, rj[0], rj[1])), (1, (1, rh[0], rh[1])), (2, (0, 1, rj[2])),
                             (4, (0, 1, rh[2])), (3, (0, 0, 1)), (5, (0, 0, 1))):
                total[:, c] += sum(w * q[:, i] for i, w in enumerate(terms) if w)
    scale = torch.tensor([f[0][0], f[0][1], f[1][0], f[2][0], f[1][1], f[2][1]], **F64)
    return total * scale / len(ovr)


def exact(case, seed):
    """The outputs in 64 bits, laid out as run() gives them.  None for the
    chemistry, whose sub-steps cell by cell would take minutes in plain
    torch, and for the steps of more than about 3e7 rays."""
    kind = case["kind"]
    if kind == "step":
        if np.prod(_shape(case)) * _rays_per_cell(case) > 3.0e7:
            return None
        return _exact_step(case, seed)
    if kind == "diffuse":
        return _exact_diffuse(case, seed)
    if kind == "smooth":
        return _exact_smooth(case, seed)
    if kind == "walk":
        start, end = (torch.tensor(v.astype(np.float64), device="cuda")
                      for v in _segments(case, seed))
        return _columns(_densities(case, seed), _shape(case), start, end)
    if kind == "rates":
        src, (table, which), idx, tau = _rays(case, seed)
        n3, shape = _densities(case, seed), _shape(case)
        cell = torch.tensor((idx[:, 0] * shape[1] + idx[:, 1]) * shape[2] + idx[:, 2],
                            device="cuda")
        g = _ray_rates(case, n3, cell, torch.tensor(src.astype(np.float64), device="cuda"),
                       torch.tensor(tau.astype(np.float64), device="cuda"),
                       torch.tensor(table, **F64), torch.tensor(which, device="cuda"),
                       *_cross_sections())
        return torch.zeros(len(n3), 6, **F64).index_add_(0, cell, g)
    return None
