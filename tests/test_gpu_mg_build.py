"""The multigrid hierarchy built on the device: a hierarchy rebuilt in its own
memory (PcMGDynamic, flags changing from solve to solve) against a fresh one,
bit for bit, and the dense inverse of single-level hierarchies, whose V-cycle
is the exact solve, so that CG ends at once."""
import ctypes as C

import numpy as np
import pytest

from mantaflow_amd import serve
from mantaflow_amd._abi import check, lib
from tests.helpers import GpuScene, obstacle_flags, smooth_vel

pytestmark = pytest.mark.gpu


def _solve(manta, g, f, v, p, pc):
    manta.solvePressure(flags=f, vel=v, pressure=p, cgAccuracy=1e-4, preconditioner=pc)
    st = manta.lastSolveStats(g.s)
    assert st["converged"]
    return p.toNumpy().copy(), v.toNumpy().copy(), st["iterations"]


# odd and even sides, two to five levels, coarsest levels of 8 to 980 unknowns
@pytest.mark.parametrize("shape", [(12, 11, 10), (33, 18, 21), (40, 64, 37), (66, 66, 66), (31, 200, 9), (70, 41, 1),
                                   (257, 130, 1)])
def test_rebuild_in_place(manta, oracle, shape):
    kinds = []
    for seed, frac in ((1, 0.0), (2, 0.2), (3, 0.1)):
        rng = np.random.default_rng(seed)
        flags = obstacle_flags(oracle, shape, frac, rng)
        vel = smooth_vel(rng, shape, passes=3)
        oracle.set_wall_bcs(shape, flags, vel)
        kinds.append((flags, vel))
    g = GpuScene(manta, shape)
    f, v, p = g.flags(kinds[0][0]), g.mac(), g.real()
    for flags, vel in (kinds[0], kinds[1], kinds[2], kinds[0]):
        f.fromNumpy(flags)
        v.fromNumpy(vel)
        got = _solve(manta, g, f, v, p, manta.PcMGDynamic)
        h = GpuScene(manta, shape)
        want = _solve(manta, h, h.flags(flags), h.mac(vel), h.real(), manta.PcMGStatic)
        np.testing.assert_array_equal(got[0], want[0])
        np.testing.assert_array_equal(got[1], want[1])
        assert got[2] == want[2]


# 27 to 1000 cells: one block of pivots, several, a short last one; the
# residual after one exact step is rounding (FP32 vectors: well below 1e-4)
@pytest.mark.parametrize("shape", [(5, 5, 5), (7, 6, 5), (9, 9, 9), (10, 10, 10), (30, 31, 1), (500, 2 + 1, 1)])
@pytest.mark.parametrize("frac", [0.0, 0.15])
def test_single_level_is_exact(manta, oracle, shape, frac):
    if shape[0] * shape[1] * shape[2] > 1000:
        shape = (330, 3, 1)
    rng = np.random.default_rng(5)
    flags = obstacle_flags(oracle, shape, frac, rng)
    vel = smooth_vel(rng, shape, passes=2)
    oracle.set_wall_bcs(shape, flags, vel)
    g = GpuScene(manta, shape)
    _, _, its = _solve(manta, g, g.flags(flags), g.mac(vel), g.real(), manta.PcMGStatic)
    assert its <= 2


def _memory(g):
    b = C.c_size_t()
    check(lib().mfx_scene_memory(g.s._h, C.byref(b)))
    return b.value


def test_hierarchies_held(manta, oracle):
    """The dynamic hierarchy stays for the next dynamic solve, counted in the
    scene's memory, and goes when a solve uses a hierarchy that is kept for
    its matrix, or with releaseMG."""
    shape = (48, 40, 44)
    n = 48 * 40 * 44
    rng = np.random.default_rng(6)
    flags = obstacle_flags(oracle, shape, 0.1, rng)
    vel = smooth_vel(rng, shape, passes=3)
    oracle.set_wall_bcs(shape, flags, vel)
    g = GpuScene(manta, shape)
    f, v, p = g.flags(flags), g.mac(vel), g.real()

    def after(pc):
        v.fromNumpy(vel)
        _solve(manta, g, f, v, p, pc)
        return _memory(g)

    after(manta.PcMGStatic)
    manta.releaseMG(g.s)
    none = _memory(g)
    one = after(manta.PcMGStatic)
    assert 8 * n < one - none < 64 * n
    assert after(manta.PcMGDynamic) == one and after(manta.PcMGDynamic) == one
    assert after(manta.PcMGStatic) == one
    after(manta.PcMGDynamic)
    manta.releaseMG(g.s)
    assert after(manta.PcMIC) == one  # one hierarchy, the code hash is not counted
    assert after(manta.PcMGDynamic) == 2 * one - none
    assert after(manta.PcMIC) == one
    manta.releaseMG(g.s)
    assert _memory(g) == none


@pytest.mark.parametrize("workers", [1, 2])
def test_served_dynamic_solves_keep_no_hierarchy(manta, workers):
    sess = [serve.PlumeScene(sh, seed=3 + i) for i, sh in enumerate([(24, 24, 24), (20, 31, 17), (16, 16, 16)])]
    for x in sess:
        x.pc = manta.PcMGDynamic
    trace = [serve.Request(i, 0.0, i % 3, serve.REQ_STEP) for i in range(9)]
    srv = serve.Server(sess, max_batch=8, workers=workers, memory_limit=1 << 30)
    srv.run(trace, realtime=False)
    assert all(x.steps == 3 for x in sess) and all(r.converged for r in srv.results)
    for x in sess:
        held = x.memory()
        manta.releaseMG(x.s)
        assert x.memory() == held
