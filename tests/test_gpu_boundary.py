"""GPU velocity boundary conditions (jg_constrain_velocity) against the
oracle's restatement of GridFractionalBoundaryConditionSolver3 /
GridBlockedBoundaryConditionSolver3::constrainVelocity.

Every step is FP64 in Jet's operand order (samplers, SDF gradient, friction,
extrapolation averages), so the result must be bit-identical."""
import numpy as np
import pytest

from jgtest import dev, host, jetgpu, torch_cuda
from systems import collider_scene

pytestmark = pytest.mark.gpu

BIG = np.finfo(np.float64).max


@pytest.fixture(scope="module")
def solver():
    if torch_cuda() is None:
        pytest.skip("no GPU")
    s = jetgpu.Solver(0)
    yield s
    s.close()


def run_gpu(solver, vel, sdf, h, o, motion, depth, closed, blocked):
    nz, ny, nx = sdf.shape
    solver.set_levels([(nx, ny, nz)])
    u, v, w = (dev(a) for a in vel)
    c = jetgpu.RigidCollider.make(*motion) if motion is not None else None
    solver.constrain_velocity(u, v, w, dev(sdf), tuple(h), tuple(o), c, depth, closed, blocked)
    return host(u), host(v), host(w)


def run_oracle(oracle, vel, sdf, h, o, motion, depth, closed, blocked):
    from oracle.jet_oracle import RigidCollider

    c = RigidCollider.make(*motion) if motion is not None else None
    return oracle.constrain_velocity(*vel, sdf, h, o, c, depth, closed, blocked)


@pytest.mark.parametrize("n,blocked,depth,closed,moving,seed", [
    ((16, 12, 10), False, 3, 63, True, 1), ((16, 12, 10), True, 3, 63, True, 2),
    ((20, 16, 14), False, 5, 1 | 8 | 32, True, 3), ((13, 17, 11), True, 0, 0, True, 4),
    ((33, 29, 31), True, 7, 63, False, 5), ((9, 5, 3), False, 2, 63, True, 6),
    ((64, 48, 40), True, 4, 2 | 4 | 16, True, 7), ((1, 1, 1), True, 1, 63, True, 8)])
def test_constrain_velocity_bitwise(solver, oracle, n, blocked, depth, closed, moving, seed):
    print(f"case constrain n={n} blocked={blocked} depth={depth} closed={closed}", flush=True)
    h, o, sdf, vel, motion = collider_scene(n, seed, moving=moving)
    got = run_gpu(solver, vel, sdf, h, o, motion, depth, closed, blocked)
    want = run_oracle(oracle, vel, sdf, h, o, motion, depth, closed, blocked)
    for a, b in zip(got, want):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("blocked", [False, True])
@pytest.mark.parametrize("closed", [63, 1 | 8 | 32])
def test_domain_kats_on_gpu(solver, blocked, closed):
    # Jet's ClosedDomain / OpenDomain: no collider, velocity 1, only the
    # closed walls' normal faces become 0.
    print(f"case constrain kat blocked={blocked} closed={closed}", flush=True)
    n = 10
    sdf = np.full((n, n, n), BIG)
    vel = (np.ones((n, n, n + 1)), np.ones((n, n + 1, n)), np.ones((n + 1, n, n)))
    u, v, w = run_gpu(solver, vel, sdf, (1.0, 1.0, 1.0), (-5.0, -5.0, -5.0), None, 5, closed,
                      blocked)
    want = [np.ones_like(a) for a in vel]
    walls = [(0, 2, 0, 1), (0, 2, -1, 2), (1, 1, 0, 4), (1, 1, -1, 8), (2, 0, 0, 16), (2, 0, -1, 32)]
    for comp, axis, end, bit in walls:
        if closed & bit:
            idx = [slice(None)] * 3
            idx[axis] = end
            want[comp][tuple(idx)] = 0.0
    for a, b in zip((u, v, w), want):
        assert np.array_equal(a, b)


def test_constrain_velocity_large_and_repeated(solver, oracle):
    # 128^3 cells, and a second call on the same solver (scratch reused,
    # validity masks rewritten) must give the same answer as a fresh oracle run.
    print("case constrain 128^3 twice", flush=True)
    h, o, sdf, vel, motion = collider_scene((128, 128, 128), 11)
    want = run_oracle(oracle, vel, sdf, h, o, motion, 3, 63, True)
    for _ in range(2):
        got = run_gpu(solver, vel, sdf, h, o, motion, 3, 63, True)
        for a, b in zip(got, want):
            assert np.array_equal(a, b)


def test_constrain_velocity_rejects_bad_arguments(solver):
    import ctypes as C

    solver.set_levels([(8, 8, 8)])
    hh = (C.c_double * 3)(0.0, 1.0, 1.0)
    oo = (C.c_double * 3)(0.0, 0.0, 0.0)
    lib = jetgpu.lib()
    assert lib.jg_constrain_velocity(solver.h, 0, hh, oo, None, None, None, None, None, 1, 63) != 0


@pytest.mark.parametrize("n,scene,seed", [
    ((63, 6, 5), "sphere", 21), ((64, 7, 6), "noise", 22), ((65, 5, 9), "corner", 23),
    ((129, 4, 3), "noise", 24), ((2, 1, 70), "noise", 25), ((24, 20, 18), "far", 26),
    ((30, 22, 26), "inside", 27), ((66, 9, 8), "nan", 28)])
def test_constrain_velocity_face_lists(solver, oracle, n, scene, seed):
    # The stages run over lists of the faces near the collider, made from a
    # bit per cell in words of 64: rows shorter than a word, one longer and
    # just over; scattered collider cells, a collider in a corner, one that
    # fills the grid, NaN distances, and an origin so far off that face
    # coordinates no longer resolve a cell (every face is listed then).
    print(f"case constrain lists n={n} scene={scene}", flush=True)
    far = (3e9, -2e9, 1e9) if scene == "far" else (0.1, -0.2, 0.05)
    h, o, sdf, vel, motion = collider_scene(n, seed, origin=far)
    r = np.random.default_rng(seed)
    if scene == "noise":
        sdf = np.where(r.random(sdf.shape) < 0.04, -r.random(sdf.shape), r.random(sdf.shape)) * h[0]
    elif scene == "corner":
        sdf[...] = h[0]
        sdf[-2:, -2:, -2:] = -h[0]
        sdf[0, 0, 0] = 0.0
    elif scene == "far":
        sdf = r.uniform(-1, 1, sdf.shape)
    elif scene == "inside":
        sdf = -1.0 - r.random(sdf.shape)
    elif scene == "nan":
        sdf[1, 2, 63] = np.nan
        sdf[4, 4, 4] = np.inf
    for blocked, depth in ((True, 4), (False, 1)):
        got = run_gpu(solver, vel, sdf, h, o, motion, depth, 63, blocked)
        want = run_oracle(oracle, vel, sdf, h, o, motion, depth, 63, blocked)
        for a, b in zip(got, want):
            assert np.array_equal(a, b, equal_nan=True)
