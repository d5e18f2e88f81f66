"""A step call that reports a HIP error after its kernels were enqueued leaves
the context's host state (step count, time, phi buffers, AB2 state) where the
device is, so that later calls wait for their own steps and report them.  The
error is an allocation the runtime refuses, left pending for the call to find."""
import ctypes

import numpy as np
import pytest

from mhit36_amd import MhitError, Solver, ic, step_batch
from mhit36_amd import _lib

pytestmark = pytest.mark.gpu

STEPS = 3


def _box(n, phiflag, q=0):
    _, dx = ic.grid(n)
    s = Solver(nx=n, dt=(0.02 + 0.01 * q) * dx, mu=0.01, f1=1.0, f2=0.5, f3=0.25, phiflag=phiflag, inflow=0,
               inphi=phiflag, radius=1.2, sigma=0.1, gamma_factor=1.2)
    s.init_fields()
    if phiflag:
        s.set_field(5, ic.drops(n, np.array([[3.0, 3.2, 2.9]]), 1.2, dx))
    return s


def _leave_an_error_pending():
    hip, p = ctypes.CDLL("libamdhip64.so"), ctypes.c_void_p()
    assert hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(1 << 60)) != 0


def _state(s, d):
    return (d.steps_done, d.t, d.status, d.gumax, d.cou, d.umean, d.vmean, d.wmean), \
        [s.get_field(f) for f in ((1, 2, 3, 4, 5) if s.params.phiflag else (1, 2, 3, 4))]


def _equal(a, b):
    assert a[0] == b[0]
    for f, (x, y) in enumerate(zip(a[1], b[1])):
        assert np.array_equal(x, y), f


@pytest.mark.parametrize("phiflag", [0, 1])
@pytest.mark.parametrize("n", [32, 128])
def test_step_after_an_error(n, phiflag):
    with _box(n, phiflag) as a, _box(n, phiflag) as b:
        a.step(STEPS)
        _leave_an_error_pending()
        with pytest.raises(MhitError) as e:
            b.step(STEPS)
        assert e.value.code == _lib.MHIT_ERR_HIP
        for _ in range(2):                 # the second of equal length, which the mirror of the first would satisfy
            _equal(_state(a, a.step(STEPS)), _state(b, b.step(STEPS)))


@pytest.mark.parametrize("phiflag", [0, 1])
def test_step_batch_after_an_error(phiflag):
    sizes = (32, 64, 32)
    alone = [_box(n, phiflag, q) for q, n in enumerate(sizes)]
    gang = [_box(n, phiflag, q) for q, n in enumerate(sizes)]
    try:
        for s in alone:
            s.step(STEPS)
        _leave_an_error_pending()
        with pytest.raises(MhitError) as e:
            step_batch(gang, STEPS)
        assert e.value.code == _lib.MHIT_ERR_HIP
        ds = step_batch(gang, STEPS)
        for a, b, d in zip(alone, gang, ds):
            _equal(_state(a, a.step(STEPS)), _state(b, d))
            _equal(_state(a, a.step(STEPS)), _state(b, b.step(STEPS)))
    finally:
        for s in alone + gang:
            s.close()
