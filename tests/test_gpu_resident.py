"""The one-kernel unpreconditioned CG of small grids against the general
kernels (which a solve with periodic residual replacement takes; a period
beyond the iteration limit never replaces anything) and, where its workgroups
give up waiting, through its fallback to them.

Both paths run GridCg's float operations in the same order and differ only in
the order of the FP64 sums behind the scalars, so the iterates are equal up to
a rounding of a scalar: the iteration counts must be equal (a stop decided by
one rounding of the residual norm would move them by one) and the solutions
within the tolerance the parity tests use for that difference."""
import numpy as np
import pytest

from mantaflow_amd._abi import lib
from tests.helpers import GpuScene, make_flags, smooth_vel

pytestmark = pytest.mark.gpu

# sizes around the splits: 2048, 4096 and 8192 cells (one workgroup), then
# runs of 2048 and 4096 cells, the last run short, rows longer than the grid
# is high, planes longer than a run
SHAPES = [(3, 3, 1), (64, 32, 1), (683, 3, 1), (64, 64, 1), (17, 241, 1), (128, 64, 1), (2731, 3, 1), (91, 91, 1),
          (353, 241, 1), (363, 363, 1), (512, 512, 1), (1500, 70, 1), (7, 9, 8), (16, 16, 16), (21, 20, 20), (44, 51, 38),
          (70, 60, 5)]


def _problem(oracle, shape, seed):
    rng = np.random.default_rng(seed)
    big = min(shape[:2]) >= 16
    flags = make_flags(oracle, shape, bw=0, open_bound="Y" if big else "", obstacles=3 if big else 0, rng=rng)
    vel = smooth_vel(rng, shape, 2, 1.0)
    oracle.set_wall_bcs(shape, flags, vel)
    return flags, vel


def _solve(manta, shape, flags, vel, general=False, **kw):
    g = GpuScene(manta, shape)
    f, v, p = g.flags(flags), g.mac(vel), g.real()
    g.s.mfxTrueResidualEvery = (1 << 30) if general else 0
    g.s.mfxRelTol = kw.pop("relTol", 0.0)
    manta.solvePressure(flags=f, vel=v, pressure=p, preconditioner=manta.PcNone, **kw)
    return p.toNumpy(), v.toNumpy(), manta.lastSolveStats(g.s)


def _close(a, b):
    assert a[2]["iterations"] == b[2]["iterations"] and a[2]["converged"] == b[2]["converged"], (a[2], b[2])
    assert abs(a[2]["resNorm"] - b[2]["resNorm"]) <= 1e-3 * abs(b[2]["resNorm"])
    for x, y in zip(a[:2], b[:2]):
        assert np.abs(x - y).max() <= 1e-4 * max(1e-6, np.abs(y).max())


@pytest.mark.parametrize("shape", SHAPES)
def test_resident_equals_general(manta, oracle, shape):
    flags, vel = _problem(oracle, shape, 7)
    kw = dict(cgAccuracy=1e-4, cgMaxIterFac=1.0)
    _close(_solve(manta, shape, flags, vel, **kw), _solve(manta, shape, flags, vel, general=True, **kw))


@pytest.mark.parametrize("shape", [(40, 50, 1), (120, 100, 1)])
@pytest.mark.parametrize("kw", [dict(useL2Norm=True, cgAccuracy=1e-5), dict(relTol=1e-3, cgMaxIterFac=9.0),
                                dict(cgAccuracy=1e-9, zeroPressureFixing=True), dict(cgMaxIterFac=0.0)])
def test_resident_options(manta, oracle, shape, kw):
    flags, vel = _problem(oracle, shape, 8)
    _close(_solve(manta, shape, flags, vel, **dict(kw)), _solve(manta, shape, flags, vel, general=True, **dict(kw)))


def test_resident_repeats_and_zero_rhs(manta, oracle):
    # the exchange words of one scene serve solve after solve
    shape = (150, 130, 1)
    flags, vel = _problem(oracle, shape, 9)
    g = GpuScene(manta, shape)
    f, v, p = g.flags(flags), g.mac(vel), g.real()
    first = None
    for k in range(4):
        v.fromNumpy(vel)
        manta.solvePressure(flags=f, vel=v, pressure=p, preconditioner=manta.PcNone, cgAccuracy=1e-4)
        got = p.toNumpy().copy()
        first = got if first is None else first
        np.testing.assert_array_equal(got, first)
    v.setConst(manta.vec3(0, 0, 0))
    manta.solvePressure(flags=f, vel=v, pressure=p, preconditioner=manta.PcNone, cgAccuracy=1e-4)
    assert not p.toNumpy().any()


@pytest.mark.parametrize("shape", [(150, 130, 1), (24, 26, 25)])
def test_resident_fallback(manta, oracle, shape):
    # with no time to wait a workgroup gives up; the solve runs again
    flags, vel = _problem(oracle, shape, 10)
    kw = dict(cgAccuracy=1e-4)
    want = _solve(manta, shape, flags, vel, general=True, **kw)
    wait = lib().mfx_testing_resident_wait
    import ctypes as C
    wait.restype, wait.argtypes = C.c_longlong, [C.c_longlong]
    wait(0)
    try:
        _close(_solve(manta, shape, flags, vel, **kw), want)
    finally:
        wait(-1)
    _close(_solve(manta, shape, flags, vel, **kw), want)


def test_resident_nan_diverges(manta, oracle):
    for shape in ((40, 40, 1), (120, 100, 1)):
        flags, vel = _problem(oracle, shape, 11)
        vel[shape[0] * 20 + 20] = np.nan
        with pytest.raises(RuntimeError, match="diverged"):
            _solve(manta, shape, flags, vel, cgAccuracy=1e-4)
