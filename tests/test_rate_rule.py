"""The quadrature form of the frequency integral (argot_hip_rate_rule, host
code) against the sum over all 256 bins in 64 bits: every rate of random rays
up to each spectrum's limit, for spectra of many shapes; the spectra that get
no limit; and tables the rule does not cover."""
import ctypes as C

import numpy as np
import pytest

from argot_amd import abi
from argot_amd import radiation as R
from argot_amd._lib import lib

EDGE = np.array([80.0, 25.0, 8.0])   # optical depths at the ranges' lower edges at scale 1
N1, N2, N3 = 12, 12, 20
THR = (1.0, 1.8125, 4.0)


def tables():
    freq, cs = R.freq_and_csect()
    run = abi.RunParam()
    run.freq = freq
    C.memmove(C.addressof(run.csect), C.addressof(cs), C.sizeof(cs))
    return run


def arrays(run):
    nu = np.ctypeslib.as_array(run.freq.nu).astype(np.float32).astype(np.float64)
    sig = np.array([[getattr(run.csect[k], f"csect_{s}") for k in range(abi.NGRID_NU)]
                    for s in ("HI", "HeI", "HeII")], np.float64)
    hsig = sig * np.maximum(nu - np.array(THR)[:, None], 0.0)
    return nu, sig, hsig


def rule(run, spec):
    spec = np.ascontiguousarray(spec, np.float32)
    n = len(spec)
    sig, dsig = np.zeros((3, 44), np.float32), np.zeros((3, 44), np.float32)
    w, lim = np.zeros((n, 192), np.float32), np.zeros(n, np.float32)
    nn = lib().argot_hip_rate_rule(C.byref(run), spec.ctypes.data, n, sig.ctypes.data,
                                   dsig.ctypes.data, w.ctypes.data, lim.ctypes.data)
    return nn, sig, dsig, w, lim


def spectra(nu):
    x = 6.626e-27 * 3.28e15 / 1.38066e-16 * nu
    s = {f"blackbody {t:.0e}": nu ** 3 / np.expm1(x / t) for t in (3e4, 5e4, 1e5, 2e5)}
    s |= {f"power law {a}": nu ** (a + 1.0) for a in (-4.0, -1.5, 0.0)}
    s["two temperatures"] = s["blackbody 1e+05"] + 30 * s["blackbody 3e+04"]
    cut = np.ones_like(nu)
    cut[128:] = 0.0
    s["cut off"] = cut
    return {k: (v / v.max()).astype(np.float32) for k, v in s.items()}


def columns(rng, sig, n, lam):
    """Columns [n, 3] whose largest edge optical depth is lam of EDGE."""
    k1, k2 = (int(np.argmax(sig[s] > 0)) for s in (1, 2))
    mix = rng.random((n, 3)) ** 2
    for s in range(3):
        mix[s::5] = np.eye(3)[s]
    u = mix / sig.max(1)
    edge = u @ sig[:, [0, k1, k2]] / EDGE
    return u * (lam / edge.max(1))[:, None]


def full_sum(sig, hsig, spec, t, d):
    """[n, 6]: sum_k S sigma f and S hsig f with the last bin's depth taken out."""
    tau, y = t @ sig, d @ sig
    f = np.exp(-(tau - tau[:, -1:])) * np.where(y > 1e-12, -np.expm1(-y) / np.maximum(y, 1e-300), 1)
    f = f * spec
    return np.concatenate([f @ sig.T, f @ hsig.T], 1)


def node_sum(sig, qs, qd, w, t, d):
    tau = np.concatenate([t[:, :1] @ qd[:1, :N1] - (t[:, 1:] @ sig[1:, -1])[:, None],
                          t[:, :2] @ qd[:2, N1:N1 + N2] - (t[:, 2:] @ sig[2:, -1])[:, None],
                          t @ qd[:, N1 + N2:]], 1)
    y = d @ qs
    f = np.exp(-tau) * np.where(y > 1e-12, -np.expm1(-y) / np.maximum(y, 1e-300), 1)
    rows = np.zeros((6, 44))
    o = 0
    for ns, n, at in ((1, N1, 0), (2, N2, N1), (3, N3, N1 + N2)):
        for s in range(ns):
            for h in range(2):
                rows[3 * h + s, at:at + n] = w[o:o + n]
                o += n
    return f @ rows.T / 2.0 ** 60


@pytest.mark.parametrize("name", list(spectra(np.ones(2) * [1.0, 2.0])))
def test_rule_equals_the_sum_over_bins_up_to_its_limit(name):
    run = tables()
    nu, sig, hsig = arrays(run)
    spec = spectra(nu)[name]
    nn, qs, qd, w, lim = rule(run, spec[None])
    assert nn == 44 and lim[0] >= 0.4
    rng = np.random.default_rng(3)
    n = 3000
    far = columns(rng, sig, n, lim[0] * rng.random(n) ** 0.3)
    part = rng.random((n, 1)) ** 2     # the cell's share of the far side's columns
    t, d = far * (1 - part), far * part
    want = full_sum(sig, hsig, spec.astype(np.float64), t, d)
    got = node_sum(sig, qs.astype(np.float64), qd.astype(np.float64), w[0].astype(np.float64), t, d)
    # 1e-7 of the rule itself, and the FP32 rounding of the tables and weights:
    # an optical depth of 2 to 4 where the sum comes from, times 6e-8, twice
    nz = want > 0
    err = np.abs(got[nz] - want[nz]) / want[nz]
    assert err.max() < 5e-7, err.max()
    assert not np.any(got[~nz])


def test_spectra_the_nodes_cannot_represent_get_no_limit():
    run = tables()
    line = np.zeros(256)
    line[50] = 1.0
    noise = np.random.default_rng(1).random(256)
    bad = np.ones(256)
    bad[200] = np.nan
    _, _, _, w, lim = rule(run, np.array([line, noise, np.zeros(256), bad]))
    assert lim[0] == 0.0 and lim[1] == 0.0 and lim[3] == 0.0
    assert lim[2] > 0.0 and not w[2].any()    # nothing: no weights, no error


@pytest.mark.parametrize("short", ["HeI edge at the first bins", "no HeII", "HeII hole"])
def test_tables_without_three_ranges_have_no_rule(short):
    run = tables()
    for k in range(256):
        if short == "HeI edge at the first bins" and k >= 4:
            run.csect[k].csect_HeI = 1e-18
        if short == "no HeII":
            run.csect[k].csect_HeII = 0.0
        if short == "HeII hole" and k == 180:
            run.csect[k].csect_HeII = 0.0
    nu, _, _ = arrays(run)
    nn, _, _, w, lim = rule(run, spectra(nu)["blackbody 1e+05"][None])
    assert nn == 0 and lim[0] == 0.0 and not w.any()
