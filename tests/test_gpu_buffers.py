"""Device buffers that change hands: advection makes a pooled buffer the
grid's data and puts the grid's old data into the solver's pool, a swap trades
two grids' data.  Every buffer has one owner and is freed once."""
import ctypes as C

import numpy as np
import pytest

from mantaflow_amd._abi import check, lib
from tests.helpers import GpuScene, rand_vel

pytestmark = pytest.mark.gpu


def _free_memory():
    f, t = C.c_size_t(), C.c_size_t()
    check(lib().mfx_device_memory(C.byref(f), C.byref(t)))
    return f.value


def _advected(manta, oracle, shape, kind, order):
    n = int(np.prod(shape))
    rng = np.random.default_rng(n + order)
    g = GpuScene(manta, shape)
    flags = oracle.init_domain(shape)
    oracle.fill_grid(shape, flags)
    f, v = g.flags(flags), g.mac(rand_vel(rng, n, 0.5))
    x = v if kind == "mac" else g.real(rng.uniform(0, 1, n).astype(np.float32))
    manta.advectSemiLagrange(flags=f, vel=v, grid=x, order=order)
    return g, x


def _drop(g):
    """Frees a solver and its grids now (the Python objects refer to each
    other, so the last reference would leave them to the collector)."""
    g.s.__del__()


@pytest.mark.parametrize("kind", ["real", "mac"])
@pytest.mark.parametrize("order", [1, 2])
def test_advected_solver_gives_its_memory_back(manta, oracle, kind, order):
    shape = (128, 120, 100)  # a Real grid takes 6 MB, a MAC grid 18 MB
    for _ in range(2):
        _drop(_advected(manta, oracle, shape, kind, order)[0])
    before = _free_memory()
    for _ in range(6):
        _drop(_advected(manta, oracle, shape, kind, order)[0])
    assert before - _free_memory() < 4 * 128 * 120 * 100


@pytest.mark.parametrize("kind", ["real", "mac"])
def test_solver_frees_no_buffer_of_another(manta, oracle, kind):
    """The advected grid is released before its solver; grids of another
    solver that take its place in memory keep their values when the first
    solver goes."""
    shape = (64, 60, 50)
    n = 64 * 60 * 50
    g, x = _advected(manta, oracle, shape, kind, 2)
    g.s._grids.remove(x)
    x._release()
    other = GpuScene(manta, shape)
    rng = np.random.default_rng(3)
    vals = [rng.uniform(-1, 1, n).astype(np.float32) for _ in range(6)]
    reals = [other.real(v) for v in vals]
    vvals = [rand_vel(rng, n) for _ in range(3)]
    vecs = [other.mac(v) for v in vvals]
    _drop(g)
    for _ in range(3):
        other.real(np.full(n, 7.0, np.float32))
        other.mac(np.full((n, 3), 7.0, np.float32))
    for r, v in zip(reals + vecs, vals + vvals):
        np.testing.assert_array_equal(r.toNumpy().reshape(v.shape), v)


def test_swap_between_solvers_moves_ownership(manta):
    """Grid::swap asks for equal sizes only (grid.h:226), so two solvers can
    trade buffers; each then frees what it holds."""
    shape = (128, 120, 100)
    n = 128 * 120 * 100
    check_mem = None
    for rep in range(5):
        a, b = GpuScene(manta, shape), GpuScene(manta, shape)
        x, y = a.real(np.full(n, 1.0, np.float32)), b.real(np.full(n, 2.0, np.float32))
        check(lib().mfx_grid_swap(x._h, y._h))
        _drop(a)
        c = GpuScene(manta, shape)
        z = c.real(np.full(n, 3.0, np.float32))
        np.testing.assert_array_equal(y.toNumpy(), np.full(n, 1.0, np.float32))
        np.testing.assert_array_equal(z.toNumpy(), np.full(n, 3.0, np.float32))
        _drop(b)
        _drop(c)
        if rep == 1:
            check_mem = _free_memory()
    assert check_mem - _free_memory() < 4 * n


def test_partial_sums_after_a_failed_growth(manta, oracle):
    """The buffers of partial sums grow with the first solve.  When that fails
    the old ones are gone: the next calls allocate again."""
    shape = (32, 30, 24)
    n = 32 * 30 * 24
    rng = np.random.default_rng(4)
    flags = oracle.init_domain(shape)
    oracle.fill_grid(shape, flags)
    vel, vals = rand_vel(rng, n, 0.5), rng.uniform(-1, 1, n).astype(np.float32)
    oracle.set_wall_bcs(shape, flags, vel)
    kw = dict(cgAccuracy=1e-4, preconditioner=manta.PcNone)
    out = []
    for fail in (False, True):
        g = GpuScene(manta, shape)
        f, v, p, r = g.flags(flags), g.mac(vel), g.real(), g.real(vals)
        assert r.getMaxAbs() == np.abs(vals).max()
        if fail:
            # the right-hand side is had, the partial sums are not
            lib().mfx_testing_fail_alloc(1)
            try:
                with pytest.raises(RuntimeError, match="memory"):
                    manta.solvePressure(flags=f, vel=v, pressure=p, **kw)
            finally:
                lib().mfx_testing_fail_alloc(-1)
            assert r.getMaxAbs() == np.abs(vals).max()
        manta.solvePressure(flags=f, vel=v, pressure=p, **kw)
        assert r.getMaxAbs() == np.abs(vals).max()
        out.append((p.toNumpy(), v.toNumpy()))
    np.testing.assert_array_equal(out[0][0], out[1][0])
    np.testing.assert_array_equal(out[0][1], out[1][1])


def test_grids_of_two_solvers(manta):
    """An operation on grids of two solvers (equal sizes are all that the
    reference asks for) comes after what either has queued, and before what
    either queues next."""
    shape = (160, 150, 140)
    n = 160 * 150 * 140
    a, b = GpuScene(manta, shape), GpuScene(manta, shape)
    x, v = a.real(), a.vec()
    y, w = b.real(), b.vec()
    one = manta.vec3(1, 1, 1)

    def queue():
        # some hundred microseconds of work on the first solver's stream
        x.setConst(0.0)
        v.setConst(manta.vec3(0, 0, 0))
        for _ in range(40):
            x.addConst(1.0)
            v.addConst(one)

    def copy():
        y.copyFrom(x)

    def add():
        y.add(x)

    def mult():
        y.mult(x)

    def component():
        manta.getComponent(v, y, 1)

    def back():
        manta.setComponent(x, w, 2)

    def swap():
        check(lib().mfx_grid_swap(y._h, x._h))

    for op, start, want in ((copy, 0.0, 40.0), (add, 2.0, 42.0), (mult, 0.5, 20.0), (component, 0.0, 40.0),
                            (back, 0.0, 0.0), (swap, 0.0, 40.0)):
        y.setConst(start)
        w.setConst(manta.vec3(0, 0, 0))
        queue()
        op()
        x.setConst(-1.0)
        v.setConst(manta.vec3(-1, -1, -1))
        assert (y.toNumpy() == want).all(), op.__name__
        if op is back:
            got = w.toNumpy().reshape(n, 3)
            assert (got[:, 2] == 40.0).all() and not got[:, :2].any()


def test_two_solvers_of_unequal_size(manta):
    """Component copies and resetOutflow's grids are as large as their partner."""
    a, b = GpuScene(manta, (16, 12, 10)), GpuScene(manta, (16, 12, 11))
    v, r = a.vec(), b.real()
    f = b.s.create(manta.FlagGrid)
    f.initDomain()
    small = a.real()
    for call in (lambda: manta.getComponent(v, r, 0), lambda: manta.setComponent(r, v, 0),
                 lambda: manta.resetOutflow(flags=f, real=small)):
        with pytest.raises(RuntimeError, match="different grid resolutions"):
            call()
