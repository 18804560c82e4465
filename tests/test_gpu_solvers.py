"""GPU CG and MGPCG (FP64 and mixed FP32/FP64) against the CPU oracle.

Pass criteria (the solver parity bar): relative residual <= 1e-8 and
||p - p_ref|| / ||p_ref|| <= 1e-6, with p_ref the oracle's FP64 solution of
the same system (modulo the mean on all-Neumann systems).  GPU CG follows
Jet's FdmCgSolver3 control flow, so its iteration count must match the
oracle's to within rounding (+-2).
"""
import numpy as np
import pytest

from jgtest import jetgpu, rel_err, rel_err_mean_free, torch_cuda
from systems import mg_poisson_hierarchy, poisson_helper, random_stencil

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def solver():
    if torch_cuda() is None:
        pytest.skip("no GPU")
    s = jetgpu.Solver(0)
    yield s
    s.close()


def upload_mg(solver, sys_):
    solver.set_levels([(x.shape[2], x.shape[1], x.shape[0]) for x in sys_.x])
    for l, A in enumerate(sys_.A):
        solver.upload(l, A, sys_.b[0] if l == 0 else None)


def test_cg_2x2_known_answer(solver):
    # Jet Cg.Solve (src/tests/unit_tests/cg_tests.cpp:16-55).
    A = np.zeros((1, 1, 2, 4))
    A[0, 0, 0] = (4.0, 1.0, 0.0, 0.0)
    A[0, 0, 1] = (3.0, 0.0, 0.0, 0.0)
    solver.set_levels([(2, 1, 1)])
    solver.upload(0, A, np.array([[[1.0, 2.0]]]))
    info = solver.cg(0, 0.0)
    assert info.iterations == 0 and info.last_residual == pytest.approx(np.sqrt(5.0), rel=1e-15)
    assert np.all(solver.download_x() == 0.0)
    info = solver.cg(10, 0.0)
    x = solver.download_x().ravel()
    assert x[0] == pytest.approx(1 / 11, rel=1e-14) and x[1] == pytest.approx(7 / 11, rel=1e-14)
    assert info.iterations <= 2 and info.last_residual <= 1e-15


# polls 0: one launch per step instead of the one launch these sizes
# take (the last two then take the tiled z-march: partial 64 x 8 x 16 tiles in x,
# y and z)
@pytest.mark.parametrize("polls", [1 << 20, 0])
@pytest.mark.parametrize("shape,tol", [((3, 3, 3), 1e-9), ((16, 12, 10), 1e-10), ((40, 40, 40), 1e-9),
                                       ((100, 20, 37), 1e-10), ((64, 13, 50), 1e-10)])
def test_cg_matches_oracle(solver, oracle, shape, tol, polls):
    print(f"case cg shape={shape} polls={polls}", flush=True)
    rng = np.random.default_rng(21)
    nx, ny, nz = shape
    A = random_stencil(nx, ny, nz, rng)
    b = rng.uniform(-1, 1, (nz, ny, nx))
    xo, io, ro, oko = oracle.cg_solve(A, b, 1000, tol)
    solver.set_levels([shape])
    solver.upload(0, A, b)
    solver.cg_polls(polls)
    try:
        info = solver.cg(1000, tol)
    finally:
        solver.cg_polls(1 << 20)
    x = solver.download_x()
    assert abs(int(info.iterations) - io) <= 2 and bool(info.converged) == oko
    assert info.last_residual <= tol
    assert rel_err(x, xo) <= 1e-6


def test_cg_closed_form_helper(solver):
    n = 24
    A, b = poisson_helper(n, n, n)
    solver.set_levels([(n, n, n)])
    solver.upload(0, A, b)
    info = solver.cg(1000, 1e-11)
    x = solver.download_x()
    d = x + np.arange(n)[None, :, None]
    assert info.converged and np.ptp(d) < 1e-8


def test_cg_max_iterations_false(solver):
    A, b = poisson_helper(12, 12, 12)
    solver.set_levels([(12, 12, 12)])
    solver.upload(0, A, b)
    info = solver.cg(3, 1e-14)
    assert info.iterations == 3 and not info.converged


def test_mgpcg_jet_unit_test(solver):
    # FdmMgpcgSolver3.Solve (src/tests/unit_tests/fdm_mgpcg_solver3_tests.cpp:13-60):
    # MGPCG(50, 4, 5, 5, 10, 10, 1e-4, 1.5) on 32^3 must return true.
    s = mg_poisson_hierarchy(4, 4)
    upload_mg(solver, s)
    p = jetgpu.mg_params(max_levels=4, restrict_iter=5, correct_iter=5, coarsest_iter=10,
                         final_iter=10, max_tol=1e-4, sor=1.5)
    info = solver.mgpcg(50, p)
    assert info.converged and info.last_residual <= 1e-4


def scene_system(oracle, kind, n, levels, seed):
    s = jetgpu.generate_scene_host(jetgpu.scene_desc(kind, n, seed=seed))
    markers, sys_ = oracle.sp_build_mg(s["u"], s["v"], s["w"], (1.0,) * 3, (0.0,) * 3,
                                       s["bsdf"], s["fsdf"], levels)
    return markers, sys_


@pytest.mark.parametrize("kind,n,levels", [(2, 64, 4), (3, 64, 4), (2, 128, 5)])
@pytest.mark.parametrize("precision", [jetgpu.JG_FP64, jetgpu.JG_MIXED])
def test_mgpcg_scene_matches_oracle(solver, oracle, kind, n, levels, precision):
    print(f"case mgpcg kind={kind} n={n} levels={levels} precision={precision}", flush=True)
    from oracle.jet_oracle import MgParams

    markers, s = scene_system(oracle, kind, n, levels, seed=5)
    upload_mg(solver, s)
    # FP64 reference solution of the same system (clean-mode oracle solve,
    # pinned by its true residual).
    ok, it, rel = oracle.mgpcg_clean_solve(s, MgParams.make(max_levels=levels, restrict_iter=2,
                                                             correct_iter=2, coarsest_iter=20,
                                                             final_iter=2), 100, 1e-12)
    assert ok and rel <= 1e-12
    p_ref = s.x[0].copy()
    p = jetgpu.mg_params(max_levels=levels, restrict_iter=2, correct_iter=2, coarsest_iter=20,
                         final_iter=2, max_tol=1e-12)
    o = jetgpu.gpu_options(precision=precision, stop_rule=jetgpu.JG_STOP_RELATIVE, rel_tol=1e-10)
    info = solver.mgpcg(200, p, o)
    x = solver.download_x()
    assert info.rel_residual <= 1e-8
    assert rel_err(x, p_ref) <= 1e-6
    # Non-fluid cells are identity rows with b = 0: p = 0 there up to the
    # solve tolerance (exactly 0 only when the smoother's SOR factor is 1,
    # since the V-cycle's correction reaches them and a sweep scales them by
    # 1 - omega).
    assert np.max(np.abs(x[markers[0] != 0])) <= 1e-6 * np.max(np.abs(p_ref))
    assert info.iterations <= 60


@pytest.mark.parametrize("precision", [jetgpu.JG_MIXED, jetgpu.JG_FP64])
def test_mgpcg_two_sweep_kernels_bitwise(solver, oracle, precision):
    # The solve with sweeps paired into two-sweep launches (z-marching and
    # brick kernels) gives the solve with single-sweep launches: the same
    # iterations, and x to rounding.  The V-cycles are bit-identical
    # (test_vcycle_two_sweep_kernel_bitwise), but the r.z / r.r sums differ
    # in order (a single last sweep emits them as block partials, a paired
    # one leaves them to a dot kernel); in mixed precision that one-ulp FP64
    # difference usually rounds away in the FP32 inner iterates, but not
    # always, so neither precision is compared bit for bit.
    markers, s = scene_system(oracle, 3, 128, 5, seed=9)
    upload_mg(solver, s)
    p = jetgpu.mg_params(max_levels=5, restrict_iter=2, correct_iter=2, coarsest_iter=20,
                         final_iter=2)
    out = {}
    for pairs in (-1, 1):
        o = jetgpu.gpu_options(precision=precision, stop_rule=jetgpu.JG_STOP_RELATIVE,
                               rel_tol=1e-9, sweep_pairs=pairs)
        info = solver.mgpcg(200, p, o)
        assert info.rel_residual <= 1e-8
        out[pairs] = (info.iterations, solver.download_x())
    assert out[-1][0] == out[1][0]
    assert rel_err(out[-1][1], out[1][1]) <= 1e-12


@pytest.mark.parametrize("depth", [2, 4])
def test_mgpcg_two_row_sweeps(solver, oracle, depth):
    # more tiles than CUs on a flat grid: FP64 single sweeps hold two tile rows
    # per thread; on two planes also the last one of level 0, which writes the
    # r.z / r.r partials (on four it holds one)
    print(f"case mgpcg two-row sweeps depth={depth}", flush=True)
    A, _ = poisson_helper(520, 500, depth)
    A[..., 0] += 0.05
    b = np.random.default_rng(35).uniform(-1, 1, A.shape[:3])
    solver.set_levels([(520, 500, depth), (260, 250, depth // 2)])
    solver.upload(0, A, b)
    solver.coarsen()
    p = jetgpu.mg_params(max_levels=2, restrict_iter=2, correct_iter=2, coarsest_iter=20,
                         final_iter=2)
    out = {}
    for pairs in (-1, 0, 1):
        info = solver.mgpcg(200, p, jetgpu.gpu_options(stop_rule=jetgpu.JG_STOP_RELATIVE,
                                                       rel_tol=1e-10, sweep_pairs=pairs))
        out[pairs] = (info.iterations, solver.download_x())
        assert info.rel_residual <= 1e-10
    assert out[-1][0] == out[0][0] == out[1][0]
    assert rel_err(out[-1][1], out[1][1]) <= 1e-12
    xo, _, _, ok = oracle.cg_solve(A, b, 2000, 1e-9)
    assert ok and rel_err(out[0][1], xo) <= 1e-6


def test_mgpcg_closed_sphere_singular(solver, oracle):
    # All-Neumann (config-1 geometry): compare modulo the mean.
    markers, s = scene_system(oracle, 1, 32, 3, seed=2)
    upload_mg(solver, s)
    xc, it, res, ok = oracle.cg_solve(s.A[0], s.b[0], 3000, 1e-10)
    assert ok
    p = jetgpu.mg_params(max_levels=3, restrict_iter=2, correct_iter=2, coarsest_iter=20,
                         final_iter=2, max_tol=1e-10)
    for prec in (jetgpu.JG_FP64, jetgpu.JG_MIXED):
        info = solver.mgpcg(200, p, jetgpu.gpu_options(precision=prec, stop_rule=jetgpu.JG_STOP_RELATIVE,
                                                       rel_tol=1e-10))
        x = solver.download_x()
        fluid = markers[0] == 0
        assert info.rel_residual <= 1e-8
        assert rel_err_mean_free(x, xc, fluid) <= 1e-6


@pytest.mark.parametrize("precision", [jetgpu.JG_FP64, jetgpu.JG_MIXED])
def test_mgpcg_poll_interval(solver, precision):
    # The host looks at the stop flag every check_every iterations; whichever
    # iteration of an interval stops the solve, the host sees it at the next
    # look.  A stop that goes unseen enqueues no-op iterations up to max_iter
    # (20000 of 18 launches: about a second against a millisecond).
    s = mg_poisson_hierarchy(4, 4)
    upload_mg(solver, s)
    p = jetgpu.mg_params(max_levels=4, restrict_iter=2, correct_iter=2, coarsest_iter=20,
                         final_iter=2)
    stops = set()
    for tol in (1e-2, 1e-3, 1e-4, 1e-5, 1e-6, 1e-7, 1e-8, 1e-9):
        base, want = None, None
        for every in (1, 2, 3, 4, 8, 2 ** 32 - 1):
            print(f"case poll interval precision={precision} tol={tol} every={every}", flush=True)
            # (an interval beyond max_iter: the only look is at max_iter)
            limit = 200 if every > 8 else 20000
            info = solver.mgpcg(limit, p, jetgpu.gpu_options(
                precision=precision, stop_rule=jetgpu.JG_STOP_RELATIVE, rel_tol=tol, check_every=every))
            x = solver.download_x()
            if every == 1:
                base, want = info, x
                stops.add(int(info.iterations) % 2)
            assert info.iterations == base.iterations and info.rel_residual == base.rel_residual
            assert np.array_equal(x, want)
            if every <= 8:
                assert info.solve_ms <= 10 * base.solve_ms, (every, info.solve_ms, base.solve_ms)
    assert stops == {0, 1}


def test_mgpcg_zero_rhs(solver):
    s = mg_poisson_hierarchy(4, 3)
    s.b[0][:] = 0.0
    upload_mg(solver, s)
    info = solver.mgpcg(10, jetgpu.mg_params(max_levels=3))
    assert info.iterations == 0 and info.converged
    assert np.all(solver.download_x() == 0.0)


def test_mgpcg_nonfinite_rhs_is_an_error(solver):
    s = mg_poisson_hierarchy(4, 2)
    s.b[0][0, 0, 0] = np.nan
    upload_mg(solver, s)
    with pytest.raises(jetgpu.JgError):
        solver.mgpcg(10, jetgpu.mg_params(max_levels=2))


def test_mgpcg_mixed_fp32_overflow_is_an_error(solver):
    # b inside FP64's range but beyond FP32's: the FP32 inner solve meets inf, and the mixed solve
    # must report a non-finite value instead of returning x = 0 as converged.  The all-Neumann
    # system needs a b that sums to zero: Jet's +-1 rows, scaled
    s = mg_poisson_hierarchy(4, 2)
    s.b[0][:] *= 1e39
    upload_mg(solver, s)
    p = jetgpu.mg_params(max_levels=2)
    with pytest.raises(jetgpu.JgError):
        solver.mgpcg(20, p, jetgpu.gpu_options(precision=jetgpu.JG_MIXED))
    info = solver.mgpcg(100, p, jetgpu.gpu_options(precision=jetgpu.JG_FP64,
                                                    stop_rule=jetgpu.JG_STOP_RELATIVE,
                                                    rel_tol=1e-9))
    assert info.converged and info.rel_residual <= 1e-9


def test_mgpcg_mixed_refinement_limit_is_not_convergence(solver):
    # one refinement (inner tolerance 1e-4 relative) cannot reach an absolute 1e-10: Jet's bool
    # must be false, as an FP64 solve stopped at max_iter would return
    s = mg_poisson_hierarchy(4, 3)
    upload_mg(solver, s)
    p = jetgpu.mg_params(max_levels=3, restrict_iter=2, correct_iter=2, coarsest_iter=20,
                         final_iter=2, max_tol=1e-10)
    info = solver.mgpcg(200, p, jetgpu.gpu_options(precision=jetgpu.JG_MIXED, max_refine=1))
    assert info.refinements == 1 and info.last_residual > 1e-10 and not info.converged
    info = solver.mgpcg(200, p, jetgpu.gpu_options(precision=jetgpu.JG_MIXED))
    assert info.last_residual <= 1e-10 and info.converged


# One launch holds the whole CG up to two rows per thread of a 1024-thread
# block on each of 256 CUs: a block less one row, exactly one, one more, the
# last grid with one row per thread (64 x 64 x 64), the first with two, the
# last of those (1024 x 512) and the first that takes the per-kernel loop.
@pytest.mark.parametrize("shape", [(33, 31, 1), (32, 32, 1), (25, 41, 1), (64, 64, 64), (65, 64, 64),
                                   (1024, 512, 1), (1024, 513, 1)])
def test_cg_one_launch_matches_oracle(solver, oracle, shape):
    print(f"case cg one launch shape={shape}", flush=True)
    rng = np.random.default_rng(31)
    nx, ny, nz = shape
    A, _ = poisson_helper(nx, ny, nz)
    A[..., 0] += 0.02  # some hundred iterations: past the 50-iteration refreshes
    b = rng.uniform(-1, 1, (nz, ny, nx))
    xo, io, ro, oko = oracle.cg_solve(A, b, 600, 1e-8)
    solver.set_levels([shape])
    solver.upload(0, A, b)
    info = solver.cg(600, 1e-8)
    x = solver.download_x()
    assert io > 50 and abs(int(info.iterations) - io) <= 2 and bool(info.converged) == oko
    # both stop at ||r|| <= 1e-8, and the smallest eigenvalue is 0.02
    assert np.linalg.norm((x - xo).ravel()) <= 2 * 1e-8 / 0.02
    again = solver.cg(600, 1e-8)
    assert again.iterations == info.iterations and np.array_equal(solver.download_x(), x)
    assert solver.cg(37, 0.0).iterations == 37


@pytest.mark.parametrize("shape", [(64, 64, 64), (65, 64, 64), (120, 100, 90), (1024, 512, 1)])
def test_cg_wait_that_runs_out_is_no_error(shape):
    # a block that gives up after two polls: every block leaves, and the solve
    # starts again as the loop of one launch per step (the third grid in its box)
    print(f"case cg wait runs out shape={shape}", flush=True)
    nx, ny, nz = shape
    A, _ = poisson_helper(nx, ny, nz)
    A[..., 0] += 0.02
    b = np.random.default_rng(33).uniform(-1, 1, (nz, ny, nx))
    if shape == (120, 100, 90):
        A[:, :, 48:, 0], A[:, :, 48:, 1:], A[:, :, 47, 1], b[:, :, 48:] = 1.0, 0.0, 0.0, 0.0
    s = jetgpu.Solver(0)
    try:
        s.set_levels([shape])
        s.upload(0, A, b)
        s.cg_polls(0)
        want = s.cg(600, 1e-8)
        x = s.download_x()
        s.cg_polls(1)
        for _ in range(2):  # the one that fails, and the next, which does not try
            info = s.cg(600, 1e-8)
            assert info.converged and info.iterations == want.iterations
            assert info.rel_residual == want.rel_residual
            assert np.array_equal(s.download_x(), x)
    finally:
        s.close()


def test_cg_one_launch_from_two_threads(solver):
    # one-launch solves of two solvers at once: each equals its
    # solve alone, bit for bit
    import threading

    print("case cg one launch, two threads", flush=True)
    rng = np.random.default_rng(32)
    out, want = [None, None], []
    solvers = [jetgpu.Solver(0) for _ in range(2)]
    try:
        for q, s in enumerate(solvers):
            A = random_stencil(64, 60, 64 + 8 * q, rng)
            s.set_levels([(64, 60, 64 + 8 * q)])
            s.upload(0, A, rng.uniform(-1, 1, A.shape[:3]))
            s.cg(300, 0.0)
            want.append(s.download_x())

        def work(q):
            for _ in range(10):
                solvers[q].cg(300, 0.0)
            out[q] = solvers[q].download_x()

        ts = [threading.Thread(target=work, args=(q,)) for q in range(2)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        assert np.array_equal(out[0], want[0]) and np.array_equal(out[1], want[1])
    finally:
        for s in solvers:
            s.close()
