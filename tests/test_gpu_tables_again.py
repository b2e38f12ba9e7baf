"""send_run_param_data with the tables changed, changed back and left as they
are: every step equals that of a context made with the tables in use."""
import ctypes as C

import numpy as np
import pytest

from argot_amd import radiation as R
from argot_amd._lib import check, lib
from helpers import small_workload

pytestmark = pytest.mark.gpu


def send(step):
    lib().send_run_param_data(C.byref(step.run), C.byref(step.cmem), C.byref(step.cpar))
    check("send_run_param_data")


def scale_tables(run, by):
    for k in range(256):
        run.csect[k].csect_HI *= by
        run.csect[k].csect_HeI *= by


def test_tables_sent_again(require_gpu):
    w = small_workload(n=16, nsrc=5, seed=91)
    a, b = R.PointSourceStep(w), R.PointSourceStep(w)
    scale_tables(b.run, 0.5)
    send(b)
    want = []
    for s in (a, b):
        s.step()
        want.append(s.rates())
    assert not np.array_equal(want[0], want[1])
    for now in (0, 0, 1, 1, 0, 1):
        C.memmove(C.addressof(a.run.csect), C.addressof(b.run.csect), C.sizeof(b.run.csect))
        if now == 0:
            scale_tables(a.run, 2.0)
        send(a)
        a.step()
        np.testing.assert_array_equal(a.rates(), want[now])
