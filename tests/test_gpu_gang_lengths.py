"""Gangs at the lengths with a factor 3 whose FFT passes are compiled for gang
launches (36 and 54: the plane passes; 72 and 108: the x and y passes; 54: a
length that takes two lines per wavefront in the projection), each box
bit-identical to the same box stepped alone; and the marches with the phase
field at tiles that do not divide the length, bit-identical to the oracle."""
import numpy as np
import pytest

from oracle import orc

from test_gpu_batch import check_gang
from test_gpu_small_boxes import _case, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("phiflag,precision", [(1, 0), (1, 1), (0, 0), (0, 1)])
@pytest.mark.parametrize("n", [36, 54, 72, 108])
def test_gang_equals_alone(n, phiflag, precision):
    check_gang(n, phiflag, precision, nbox=2, nsteps=3, forced=True)


@pytest.mark.parametrize("n", [108, 162])
def test_marches_with_phase_field_equal_the_oracle(n):
    kw, fields = _case(n, 1, 0)
    got = _run(kw, fields, steps=2)
    o = orc.Oracle(**kw)
    for f, a in fields.items():
        o.set_field(f, a)
    o.step(2)
    for f, a in got.items():
        assert np.array_equal(a, o.get_field(f)), f
    o.close()
