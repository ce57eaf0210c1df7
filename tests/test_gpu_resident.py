"""The one-kernel unpreconditioned CG of small grids against the general
kernels (which a solve with periodic residual replacement takes; a period
beyond the iteration limit never replaces anything) and, where its workgroups
give up waiting, through its fallback to them.

Both paths run GridCg's float operations in the same order and differ only in
the order of the FP64 sums behind the scalars, so the iterates are equal up to
a rounding of a scalar: the iteration counts must be equal (a stop decided by
one rounding of the residual norm would move them by one) and the solutions
within the tolerance the parity tests use for that difference."""
import ctypes as C
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from contextlib import contextmanager

import numpy as np
import pytest

from mantaflow_amd._abi import lib
from tests.helpers import GpuScene, make_flags, smooth_vel

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

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
    before = _counts()
    with _hook("mfx_testing_resident_wait", C.c_longlong(0), -1):
        got = _solve(manta, shape, flags, vel, **kw)
    assert _counts() == (before[0] + 1, before[1] + 1)
    _close(got, want)
    np.testing.assert_array_equal(got[0], want[0])
    _close(_solve(manta, shape, flags, vel, **kw), want)
    assert _counts() == (before[0] + 2, before[1] + 1)


def test_resident_tags_wrap(manta, oracle):
    """The words carry 32-bit tags; before they run out the words are cleared
    and the count starts again.  The solve that ends at the last tag and the
    ones after it give the bits of the first."""
    shape = (150, 130, 1)
    flags, vel = _problem(oracle, shape, 15)
    g = GpuScene(manta, shape)
    f, v, p = g.flags(flags), g.mac(vel), g.real()
    tag = lib().mfx_testing_resident_next
    tag.restype, tag.argtypes = C.c_uint, [C.c_void_p, C.c_uint]
    seen, out = [], []
    for k in range(4):
        if k == 1:
            need = seen[0] - 1  # tags of one solve
            tag(g.s._h, 2 ** 32 - 1 - need)
        v.fromNumpy(vel)
        before = _counts()
        manta.solvePressure(flags=f, vel=v, pressure=p, preconditioner=manta.PcNone, cgAccuracy=1e-4)
        assert _counts() == (before[0] + 1, before[1])
        seen.append(tag(g.s._h, 0))
        out.append(p.toNumpy().copy())
    assert seen[1] == 2 ** 32 - 1 and seen[2] == 1 + need and seen[3] == 1 + 2 * need
    for o in out[1:]:
        np.testing.assert_array_equal(o, out[0])


def test_resident_nan_diverges(manta, oracle):
    for shape in ((40, 40, 1), (120, 100, 1)):
        flags, vel = _problem(oracle, shape, 11)
        vel[shape[0] * 20 + 20] = np.nan
        with pytest.raises(RuntimeError, match="diverged"):
            _solve(manta, shape, flags, vel, cgAccuracy=1e-4)


def _counts():
    """(one-kernel solves queued, of them given up) so far"""
    a, b = C.c_longlong(), C.c_longlong()
    lib().mfx_testing_resident_counts(C.byref(a), C.byref(b))
    return a.value, b.value


def _launches():
    f = lib().mfx_testing_resident_launches
    f.restype = C.c_longlong
    return f()


@contextmanager
def _hook(name, value, back):
    f = getattr(lib(), name)
    f.argtypes = [type(value)]
    f(value)
    try:
        yield
    finally:
        f(type(value)(back))


def test_resident_needs_a_unit_per_workgroup(manta, oracle):
    # 150x130 cells are 10 workgroups, 60x60 one (which waits for nobody)
    shape, small = (150, 130, 1), (60, 60, 1)
    flags, vel = _problem(oracle, shape, 12)
    sflags, svel = _problem(oracle, small, 12)
    kw = dict(cgAccuracy=1e-4)
    want = _solve(manta, shape, flags, vel, general=True, **kw)
    for cus, ran in ((9, 0), (10, 1), (64, 1)):
        with _hook("mfx_testing_resident_cus", C.c_int(cus), 0):
            before = _counts()
            _close(_solve(manta, shape, flags, vel, **kw), want)
            assert _counts() == (before[0] + ran, before[1]), cus
    with _hook("mfx_testing_resident_cus", C.c_int(1), 0):
        before = _counts()
        _solve(manta, small, sflags, svel, **kw)
        assert _counts() == (before[0] + 1, before[1])


def test_resident_rests_after_giving_up(manta, oracle):
    shape = (150, 130, 1)
    flags, vel = _problem(oracle, shape, 10)
    kw = dict(preconditioner=manta.PcNone, cgAccuracy=1e-4)
    g = GpuScene(manta, shape)
    f, v, p = g.flags(flags), g.mac(vel), g.real()

    def solve():
        v.fromNumpy(vel)
        before = _counts()
        manta.solvePressure(flags=f, vel=v, pressure=p, **kw)
        after = _counts()
        return p.toNumpy().copy(), (after[0] - before[0], after[1] - before[1])

    whole = solve()
    assert whole[1] == (1, 0)
    with _hook("mfx_testing_resident_wait", C.c_longlong(0), -1):
        gave = solve()
        assert gave[1] == (1, 1)
    # the wait was paid once: this solver's next solves do not try again
    for _ in range(3):
        again = solve()
        assert again[1] == (0, 0)
        np.testing.assert_array_equal(again[0], gave[0])
    # another solver does
    h = GpuScene(manta, shape)
    f, v, p = h.flags(flags), h.mac(vel), h.real()
    other = solve()
    assert other[1] == (1, 0)
    np.testing.assert_array_equal(other[0], whole[0])


# by threads and cells per thread: 42, 10, 52, 42, 10, 52 workgroups, 64, 33,
# 64, 33 and twice one; a launch holds as many as there are units (256)
@pytest.mark.parametrize("cus,launches", [(0, 3), (64, 9)])
def test_resident_solves_at_once(manta, oracle, cus, launches):
    """A batch's unpreconditioned problems share launches, as many as the
    device (or 64 units of it) holds at once, and give the bits of solves
    alone."""
    shapes = [(353, 241, 1), (512, 512, 1), (150, 130, 1), (64, 64, 1), (363, 363, 1), (1500, 70, 1)] * 2
    kw = dict(preconditioner=manta.PcMIC, cgAccuracy=1e-4)
    single, batch = [], []
    for k, shape in enumerate(shapes):
        flags, vel = _problem(oracle, shape, 20 + k)
        for out in (single, batch):
            g = GpuScene(manta, shape)
            out.append((g, g.flags(flags), g.mac(vel), g.real()))
    for g, f, v, p in single:
        manta.solvePressure(flags=f, vel=v, pressure=p, **kw)
    with _hook("mfx_testing_resident_cus", C.c_int(cus), 0):
        before, n = _counts(), _launches()
        manta.solvePressureBatch([(v, p, f) for g, f, v, p in batch], **kw)
        assert _counts() == (before[0] + len(shapes), before[1])
        assert _launches() - n == launches
    for (g1, f1, v1, p1), (g2, f2, v2, p2) in zip(single, batch):
        assert manta.lastSolveStats(g1.s)["iterations"] == manta.lastSolveStats(g2.s)["iterations"]
        np.testing.assert_array_equal(p1.toNumpy(), p2.toNumpy())
        np.testing.assert_array_equal(v1.toNumpy(), v2.toNumpy())


@pytest.mark.parametrize("cus", [0, 128, 64])
def test_resident_solves_on_threads(manta, oracle, cus):
    """Solvers on threads of their own, each on its own stream, solve at once,
    again and again: more workgroups than fit together (297; counted with 128
    and 64 units two solves and one at a time).  None gives up waiting and each
    result is that of the solve alone."""
    shapes = [(353, 241, 1), (512, 512, 1), (150, 130, 1), (363, 363, 1), (1500, 70, 1), (70, 60, 40), (48, 48, 48)]
    work = []
    for k, shape in enumerate(shapes):
        flags, vel = _problem(oracle, shape, 80 + k)
        g = GpuScene(manta, shape)
        f, v, p = g.flags(flags), g.mac(vel), g.real()

        def solve(f=f, v=v, p=p, vel=vel):
            v.fromNumpy(vel)
            manta.solvePressure(flags=f, vel=v, pressure=p, preconditioner=manta.PcNone, cgAccuracy=1e-4)
            return p.toNumpy().copy(), v.toNumpy().copy()
        work.append((g, solve, solve()))
    with _hook("mfx_testing_resident_cus", C.c_int(cus), 0):
        before = _counts()
        with ThreadPoolExecutor(len(work)) as ex:
            runs = [ex.submit(lambda s=solve: [s() for _ in range(4)]) for _, solve, _ in work]
            got = [r.result(timeout=60) for r in runs]
        assert _counts() == (before[0] + 4 * len(work), before[1])
    for (_, _, want), out in zip(work, got):
        for o in out:
            np.testing.assert_array_equal(o[0], want[0])
            np.testing.assert_array_equal(o[1], want[1])


@pytest.mark.parametrize("relTol", [0.0, 1e-3])
def test_resident_beside_iterated_problems(manta, oracle, relTol):
    """One-kernel problems first, last and among problems with a preconditioner
    and an unpreconditioned one too large for it: each as alone."""
    shapes = [(40, 40, 1), (24, 22, 20), (150, 130, 1), (33, 30, 28), (800, 700, 1), (90, 90, 1), (64, 64, 1)]
    kw = dict(preconditioner=manta.PcMIC, cgAccuracy=1e-3)
    single, batch = [], []
    for k, shape in enumerate(shapes):
        flags, vel = _problem(oracle, shape, 60 + k)
        for out in (single, batch):
            g = GpuScene(manta, shape)
            g.s.mfxRelTol = relTol
            out.append((g, g.flags(flags), g.mac(vel), g.real()))
    for g, f, v, p in single:
        manta.solvePressure(flags=f, vel=v, pressure=p, **kw)
    manta.solvePressureBatch([(v, p, f) for g, f, v, p in batch], **kw)
    for (g1, f1, v1, p1), (g2, f2, v2, p2) in zip(single, batch):
        s1, s2 = manta.lastSolveStats(g1.s), manta.lastSolveStats(g2.s)
        for key in ("iterations", "resNorm", "relResidual", "converged"):
            assert s1[key] == s2[key], (key, s1, s2)
        np.testing.assert_array_equal(p1.toNumpy(), p2.toNumpy())
        np.testing.assert_array_equal(v1.toNumpy(), v2.toNumpy())


def test_resident_batch_fallback(manta, oracle):
    """Workgroups of a batch's problems that give up: those problems run again
    on the general kernels, the others are not touched."""
    shapes = [(150, 130, 1), (64, 64, 1), (24, 24, 24), (353, 241, 1)]
    kw = dict(preconditioner=manta.PcMIC, cgAccuracy=1e-4)
    want, batch = [], []
    for k, shape in enumerate(shapes):
        flags, vel = _problem(oracle, shape, 40 + k)
        many = shape[2] == 1 and shape != (64, 64, 1)
        want.append(_solve(manta, shape, flags, vel, general=True, cgAccuracy=1e-4) if many else None)
        for out in (batch, None):
            g = GpuScene(manta, shape)
            f, v, p = g.flags(flags), g.mac(vel), g.real()
            if out is None and not many:
                manta.solvePressure(flags=f, vel=v, pressure=p, **kw)
                want[-1] = p.toNumpy(), v.toNumpy(), manta.lastSolveStats(g.s)
            elif out is not None:
                out.append((g, f, v, p))
    with _hook("mfx_testing_resident_wait", C.c_longlong(0), -1):
        before = _counts()
        manta.solvePressureBatch([(v, p, f) for g, f, v, p in batch], **kw)
        assert _counts() == (before[0] + 3, before[1] + 2)
    for (g, f, v, p), w in zip(batch, want):
        _close((p.toNumpy(), v.toNumpy(), manta.lastSolveStats(g.s)), w)


def test_resident_limit_is_per_wait(manta, oracle):
    """The limit bounds one wait (a few microseconds), not the solve: one that
    runs several times as long as the limit of 1 ms is not given up."""
    shape = (353, 241, 1)
    flags, vel = _problem(oracle, shape, 13)
    with _hook("mfx_testing_resident_wait", C.c_longlong(100000), -1):
        before = _counts()
        got = _solve(manta, shape, flags, vel, cgAccuracy=2e-7, cgMaxIterFac=3.0)
        assert _counts() == (before[0] + 1, before[1])
    assert got[2]["seconds"] > 4 * 1e-3, got[2]


def test_resident_without_its_words(manta, oracle):
    """The exchange words are the one buffer the general kernels do not need:
    without them the solve runs on those, and takes the words when it can."""
    shape = (150, 130, 1)
    flags, vel = _problem(oracle, shape, 14)
    g = GpuScene(manta, shape)
    f, v, p = g.flags(flags), g.mac(vel), g.real()
    out = []
    for every, after, ran in (((1 << 30), -1, 0), (0, 0, 0), (0, -1, 1)):
        v.fromNumpy(vel)
        g.s.mfxTrueResidualEvery = every
        before = _counts()
        lib().mfx_testing_fail_alloc(after)
        try:
            manta.solvePressure(flags=f, vel=v, pressure=p, preconditioner=manta.PcNone, cgAccuracy=1e-4)
        finally:
            lib().mfx_testing_fail_alloc(-1)
        assert _counts()[0] - before[0] == ran
        out.append((p.toNumpy().copy(), v.toNumpy().copy(), dict(manta.lastSolveStats(g.s))))
    np.testing.assert_array_equal(out[1][0], out[0][0])
    _close(out[2], out[0])


def test_resident_beside_another_runtime():
    """torch loads a HIP runtime of its own; the one-kernel CG runs all the same
    (in a child process, so that the other tests keep one runtime)."""
    prog = """
import ctypes as C
from mantaflow_amd import manta
import torch
from mantaflow_amd._abi import lib
s = manta.Solver(name="t", gridSize=manta.vec3(150, 130, 1), dim=2)
f, v, p = s.create(manta.FlagGrid), s.create(manta.MACGrid), s.create(manta.RealGrid)
f.initDomain()
f.fillGrid()
v.setConst(manta.vec3(0.1, 0.2, 0))
manta.setWallBcs(flags=f, vel=v)
manta.solvePressure(flags=f, vel=v, pressure=p, preconditioner=manta.PcNone, cgAccuracy=1e-4)
ran, gave = C.c_longlong(), C.c_longlong()
lib().mfx_testing_resident_counts(C.byref(ran), C.byref(gave))
print("counts", ran.value, gave.value)
"""
    r = subprocess.run([sys.executable, "-c", prog], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "counts 1 0" in r.stdout, r.stdout + r.stderr
