"""Launch shapes on the host: for every accepted length, every shape that a knob
takes gives a launch the device accepts in each use of it (a box stepped alone,
a gang, the turbulent start), whose kernels may be of different forms."""
import ctypes

import pytest

from mhit36_amd import _lib

KNOBS = _lib.KNOBS
MARCH, REGS, LDS, SMALL = range(4)
LENGTHS = sorted(2 ** a * 3 ** b for a in range(1, 12) for b in range(7) if 4 <= 2 ** a * 3 ** b <= 2048)


def launch(n, precision, use, knob, **shapes):
    """(form, shape, threads, lds) or None for a shape the knob does not take."""
    value, out = (ctypes.c_int * len(KNOBS))(), (ctypes.c_int * 4)()
    for k, v in shapes.items():
        value[KNOBS.index(k)] = v
    rc = _lib.load().mhit_debug_launch_shape(n, precision, use, value, KNOBS.index(knob), out)
    if rc == _lib.MHIT_ERR_ARG:
        return None
    assert rc == _lib.MHIT_OK, (n, precision, use, knob, shapes, rc)
    return tuple(out)


def least_radix(n):
    a = (n & -n).bit_length() - 1
    return 2 if a == 1 else 3 if n % 3 == 0 else 8 if a % 3 == 0 else 4


@pytest.mark.parametrize("precision", [0, 1])
def test_every_shape_fits_every_use(precision):
    bad = []
    for n in LENGTHS:
        for knob in KNOBS:
            for v in [0] + [2 ** q for q in range(11)]:
                alone = launch(n, precision, 0, knob, **{knob: v})
                for use in (0, 1, 2):
                    got = launch(n, precision, use, knob, **{knob: v})
                    assert (got is None) == (alone is None), (n, knob, v, use)
                    if got is None:
                        continue
                    form, lines, threads, lds = got
                    ok = 64 <= threads <= 1024 or (form == REGS and 1 <= threads <= 1024)
                    ok = ok and lds <= 163840 and (form == SMALL or lines >= 1)
                    if form == LDS:                  # one butterfly of the smallest radix per thread
                        ok = ok and threads * least_radix(n) >= lines * n
                    if not ok:
                        bad.append((n, knob, v, use) + got)
    assert not bad, bad


@pytest.mark.parametrize("precision", [0, 1])
def test_a_shape_set_by_hand_is_the_one_that_runs(precision):
    """Small boxes run forms without a shape, unless one is set by hand: then
    the pass that has it runs, with that shape, also where it is the default."""
    small = set()
    for n in LENGTHS:
        for knob in KNOBS:
            if launch(n, precision, 0, knob)[0] == SMALL:
                small.add((knob, n))
            for v in [2 ** q for q in range(11)]:
                got = launch(n, precision, 0, knob, **{knob: v})
                if got:
                    assert got[0] == MARCH if knob.startswith("kz") else got[0] in (REGS, LDS), (n, knob, v, got)
                    assert got[1] == v, (n, knob, v, got)
    sizes = {knob: [n for k, n in sorted(small) if k == knob] for knob in KNOBS}
    assert sizes["kz_phase"] == [n for n in LENGTHS if n <= 72]
    assert sizes["kz_momentum"] == [n for n in LENGTHS if n <= (96 if precision else 64)]
    assert sizes["xinv_pairs"] == [32, 36, 48, 54, 64] and not sizes["z_tile"]


def test_unknown_lengths_and_shapes_are_refused():
    value, out = (ctypes.c_int * len(KNOBS))(), (ctypes.c_int * 4)()
    lib = _lib.load()
    for n in (0, 2, 7, 10, 50, 4096):
        assert lib.mhit_debug_launch_shape(n, 0, 0, value, 0, out) == _lib.MHIT_ERR_BAD_N
    assert lib.mhit_debug_launch_shape(32, 2, 0, value, 0, out) == _lib.MHIT_ERR_UNSUPPORTED
    assert lib.mhit_debug_launch_shape(32, 0, 3, value, 0, out) == _lib.MHIT_ERR_ARG
    assert lib.mhit_debug_launch_shape(32, 0, 0, None, 0, out) == _lib.MHIT_ERR_ARG
    assert launch(32, 0, 0, "kz_momentum", kz_momentum=3) is None
    assert launch(32, 0, 0, "y_tile", y_tile=1024) is None


@pytest.mark.gpu
@pytest.mark.parametrize("n,precision", [(432, 0), (486, 1)])
def test_default_shapes_by_hand_run_every_use(n, precision):
    """The lengths whose default column tile fits the one-box kernels alone: the
    turbulent start and a gang of a box that holds the defaults as shapes set by
    hand give what a box left to its defaults gives, bit for bit."""
    import numpy as np
    from mhit36_amd import Solver, step_batch

    dx = 2 * np.pi / (n - 1)
    kw = dict(nx=n, dt=0.06 * dx, mu=0.002, f1=1.0, f2=1.0, f3=1.0, phiflag=0, inflow=1, precision=precision)
    with Solver(**kw) as a, Solver(**kw) as b:
        b.set_tuning(**{k: v for k, v in b.tuning()["heuristic"].items() if k != "kz_phase"})
        for s in (a, b):
            s.init_random_velocity(seed=17, k_peak=4.0, urms=1.0)
        for f in (1, 2, 3):
            assert np.array_equal(a.get_field(f), b.get_field(f)), f
        da, (db,) = a.step(2), step_batch([b], 2)
        assert (da.steps_done, da.gumax, da.cou) == (2, db.gumax, db.cou)
        for f in (1, 2, 3, 4):
            assert np.array_equal(a.get_field(f), b.get_field(f)), f
