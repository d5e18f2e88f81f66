"""The marching momentum pass at ragged tiles and at slab heights of two
planes and of all that the length allows: FP64 bit-identical to the oracle, FP32
state to the one-point form that these sizes take by default."""
import numpy as np
import pytest

from oracle import orc

from test_gpu_small_boxes import _case, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("phiflag", [0, 1])
@pytest.mark.parametrize("n", [4, 16, 18, 36, 48, 54, 64, 72])
def test_march_equals_the_oracle(n, phiflag):
    kw, fields = _case(n, phiflag, 0)
    o = orc.Oracle(**kw)
    for f, a in fields.items():
        o.set_field(f, a)
    o.step(3)
    for kz in sorted({2, n & -n}):
        for f, a in _run(kw, fields, kz_momentum=kz).items():
            assert np.array_equal(a, o.get_field(f)), (kz, f)
    o.close()


@pytest.mark.parametrize("phiflag", [0, 1])
@pytest.mark.parametrize("n", [16, 36, 54, 64, 96])
def test_mixed_march_equals_the_point_form(n, phiflag):
    kw, fields = _case(n, phiflag, 1)
    want = _run(kw, fields)
    for kz in sorted({2, n & -n}):
        for f, a in _run(kw, fields, kz_momentum=kz).items():
            assert np.array_equal(a, want[f]), (kz, f)
