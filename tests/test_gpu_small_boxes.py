"""The forms of the phase-field and momentum passes that small boxes take (no
march along z): bit-identical to the oracle in FP64, and to the marching forms
in mixed precision.  Sizes below, at and above a tile in each direction, ragged
ones, and the first sizes past each form's range."""
import numpy as np
import pytest

from mhit36_amd import Solver, ic
from oracle import orc

from gpu_util import random_velocity

pytestmark = pytest.mark.gpu


def _case(n, phiflag, precision):
    u, v, w = random_velocity(n, seed=n)
    _, dx = ic.grid(n)
    fields = {1: u, 2: v, 3: w}
    if phiflag:
        fields[5] = ic.drops(n, np.array([[3.0, 3.2, 2.9]]), 1.2, dx)
    kw = dict(nx=n, dt=0.002 * dx, mu=0.01, f1=0.7, f2=0.5, f3=0.3, k0=2.0, phiflag=phiflag, inflow=1,
              inphi=phiflag, radius=1.2, sigma=0.1, gamma_factor=1.2, precision=precision)
    return kw, fields


def _run(kw, fields, steps=3, **shapes):
    with Solver(**kw) as s:
        s.set_tuning(**shapes)
        for f, a in fields.items():
            s.set_field(f, a)
        s.step(steps)
        return {f: s.get_field(f) for f in (1, 2, 3, 4) + ((5,) if kw["phiflag"] else ())}


@pytest.mark.parametrize("phiflag", [0, 1])
@pytest.mark.parametrize("n", [4, 8, 16, 18, 32, 36, 54, 64, 72, 96])
def test_small_boxes_equal_the_oracle(n, phiflag):
    kw, fields = _case(n, phiflag, 0)
    got = _run(kw, fields)
    o = orc.Oracle(**kw)
    for f, a in fields.items():
        o.set_field(f, a)
    o.step(3)
    for f, a in got.items():
        assert np.array_equal(a, o.get_field(f)), f
    o.close()


@pytest.mark.parametrize("phiflag", [0, 1])
@pytest.mark.parametrize("n", [16, 32, 48, 64, 72, 96, 108])
def test_small_boxes_mixed_equal_the_marches(n, phiflag):
    kw, fields = _case(n, phiflag, 1)
    with Solver(**kw) as s:
        h = s.tuning()["heuristic"]
    other = {k: 4 if h[k] != 4 else 2 for k in ("kz_phase", "kz_momentum")}
    a, b = _run(kw, fields), _run(kw, fields, **other)
    for f in a:
        assert np.array_equal(a[f], b[f]), f
