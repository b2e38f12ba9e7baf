"""The walk's FP32 quotient (argot_hip_quotients, host code) equals IEEE
division: random operands over the walk's ranges, and the quotients that lie
closest to the middle of two floats, found for each divisor by solving
A 2^sh = B m + j for the odd 25-bit m and small j."""
import numpy as np
import pytest

from argot_amd._lib import lib


def check(a, b):
    a, b = np.ascontiguousarray(a, np.float32), np.ascontiguousarray(b, np.float32)
    q = np.zeros_like(a)
    lib().argot_hip_quotients(a.ctypes.data, b.ctypes.data, q.ctypes.data, len(a))
    want = a / b
    bad = q.view(np.uint32) != want.view(np.uint32)
    assert not bad.any(), (a[bad][:3], b[bad][:3], q[bad][:3], want[bad][:3])


def test_random_quotients():
    rng = np.random.default_rng(1)
    n = 2_000_000
    a = (1 + rng.random(n)) * 2.0 ** rng.integers(-40, 2, n) * rng.choice([-1, 1], n)
    b = (1 + rng.random(n)) * 2.0 ** rng.integers(-12, 0, n) * rng.choice([-1, 1], n)
    check(a, b)
    # directions almost in a coordinate plane, down to the TINY guard, and zero distances
    b = (1 + rng.random(n)) * 2.0 ** rng.integers(-102, 0, n)
    a = (1 + rng.random(n)) * 2.0 ** rng.integers(-30, 0, n)
    a[::7] = 0.0
    b[::5] = 1.0e-31
    check(a, b)


@pytest.mark.parametrize("sh", [24, 25])
def test_quotients_next_to_the_middle_of_two_floats(sh):
    rng = np.random.default_rng(sh)
    B = np.concatenate([rng.integers(1 << 23, 1 << 24, 60000), (1 << 24) - 1 - np.arange(3000),
                        (1 << 23) + np.arange(3000)]).astype(np.uint64) | np.uint64(1)
    inv = B.copy()                       # 1/B modulo 2^64
    for _ in range(6):
        inv = inv * (np.uint64(2) - B * inv)
    aa, bb = [], []
    M = np.uint64((1 << sh) - 1)
    for j in range(-7, 8, 2):
        m = (inv * np.uint64(-j % (1 << 64))) & M
        for mm in (m, m + np.uint64(1 << 24)):
            A = (B.astype(object) * mm.astype(object) + j)
            ok = np.array([(x % (1 << sh) == 0) and ((1 << 23) <= (x >> sh) < (1 << 24))
                           and (1 << 24) < y < (1 << 25) and y & 1
                           for x, y in zip(A, mm.astype(object))])
            aa.append(np.array([float(x >> sh) for x in A[ok]]))
            bb.append(B[ok].astype(np.float64))
    a, b = np.concatenate(aa), np.concatenate(bb)
    assert len(a) > 50000
    check(a * 2.0 ** -24, b * 2.0 ** -24)
