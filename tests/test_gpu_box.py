"""Solves in the bounding box of the cells that take part (jg_box.h).

A system whose fluid fills part of the grid is solved on that part only.  The
reference is the same system with a right-hand side of 1e-30 in two opposite
corner cells (decoupled air cells, whose solution is then 1e-30): every cell
of the grid lies between two that take part, so that solve is of the whole
grid.  Both stop at a relative residual of 1e-8 (1e-12 for the reference), so
they agree as the oracle's solutions are required to: 1e-6."""
import numpy as np
import pytest

from jgtest import dev, empty, jetgpu, rel_err, torch_cuda

pytestmark = pytest.mark.gpu

PARAMS = dict(restrict_iter=2, correct_iter=2, coarsest_iter=20, final_iter=2, max_tol=0.0, sor=1.3)


@pytest.fixture(scope="module")
def solver():
    if torch_cuda() is None:
        pytest.skip("no GPU")
    s = jetgpu.Solver(0)
    yield s
    s.close()


def view(solver, ptr, n):
    import torch

    return torch.as_tensor(jetgpu._DeviceView(ptr, n, "<f8"), device="cuda")


def rhs(solver, shape):
    return view(solver, solver.rhs_ptr(), int(np.prod(shape))).view(*shape[::-1])


def build(solver, shape, levels, block, seed):
    """Fluid in the cells of block = ((x0, x1), (y0, y1), (z0, z1)), air elsewhere."""
    nx, ny, nz = shape
    twod = nz == 1
    solver.set_levels([(nx >> l, ny >> l, 1 if twod else nz >> l) for l in range(levels)])
    rng = np.random.default_rng(seed)
    fs = np.ones((nz, ny, nx))
    (x0, x1), (y0, y1), (z0, z1) = block
    fs[z0:z1, y0:y1, x0:x1] = -1.0
    bs = np.ones((nz, ny, nx))
    u = rng.uniform(-1, 1, (nz, ny, nx + 1))
    v = rng.uniform(-1, 1, (nz, ny + 1, nx))
    if twod:
        solver.sp_build2(dev(u), dev(v), dev(bs), dev(fs), (1.0, 1.0))
    else:
        w = rng.uniform(-1, 1, (nz + 1, ny, nx))
        solver.sp_build(dev(u), dev(v), dev(w), dev(bs), dev(fs), 1.0)
    return fs < 0


def solve(solver, levels, precision, tol=1e-8):
    info = solver.mgpcg(300, jetgpu.mg_params(max_levels=levels, **PARAMS),
                        jetgpu.gpu_options(precision=precision, stop_rule=jetgpu.JG_STOP_RELATIVE,
                                           rel_tol=tol))
    return solver.download_x(), info


# the block at the origin, in the far corner, floating (and not aligned to the
# coarsest cells), a thin slab, and two one-plane grids
@pytest.mark.parametrize("shape,levels,block", [
    ((96, 80, 64), 4, ((0, 50), (0, 40), (0, 64))),
    ((96, 80, 64), 4, ((41, 96), (33, 80), (9, 64))),
    ((72, 88, 80), 3, ((13, 45), (21, 62), (34, 71))),
    ((128, 64, 66), 2, ((0, 128), (30, 33), (0, 66))),
    ((640, 512, 1), 5, ((100, 333), (0, 200), (0, 1))),
    ((768, 512, 1), 1, ((700, 768), (500, 512), (0, 1)))])
@pytest.mark.parametrize("precision", [jetgpu.JG_FP64, jetgpu.JG_MIXED])
def test_box_solve_matches_whole_grid(solver, shape, levels, block, precision):
    print(f"case box shape={shape} block={block} precision={precision}", flush=True)
    fluid = build(solver, shape, levels, block, 3)
    x, info = solve(solver, levels, precision)
    assert info.converged and info.rel_residual <= 1e-8
    b = rhs(solver, shape)
    # an air cell's row is x = b = 0, so x there is the residual that is left
    assert np.linalg.norm(x[~fluid]) <= 1e-8 * float(b.norm())
    b[0, 0, 0] += 0.0 if fluid[0, 0, 0] else 1e-30
    b[-1, -1, -1] += 0.0 if fluid[-1, -1, -1] else 1e-30
    whole, iw = solve(solver, levels, jetgpu.JG_FP64, 1e-12)
    assert iw.rel_residual <= 1e-12
    assert rel_err(x, whole) <= 1e-6
    again, i2 = solve(solver, levels, precision)  # whole grid, the same tolerance
    assert abs(int(i2.iterations) - int(info.iterations)) <= 4
    # and the next system, smaller: the box follows the system
    build(solver, shape, levels, ((0, 8), (0, 8), (0, min(8, shape[2]))), 4)
    x, info = solve(solver, levels, precision)
    assert info.converged and info.rel_residual <= 1e-8


@pytest.mark.parametrize("shape,block", [((48, 40, 41), ((3, 30), (11, 40), (5, 33))),
                                         ((120, 100, 90), ((0, 100), (20, 75), (0, 90))),
                                         ((300, 230, 1), ((17, 200), (0, 131), (0, 1)))])
def test_box_cg_matches_whole_grid(solver, shape, block):
    print(f"case box cg shape={shape}", flush=True)
    fluid = build(solver, shape, 1, block, 5)
    info = solver.cg(3000, 1e-9)
    x = solver.download_x()
    assert info.converged and np.all(x[~fluid] == 0.0)
    b = rhs(solver, shape)
    b[0, 0, 0] += 0.0 if fluid[0, 0, 0] else 1e-30
    b[-1, -1, -1] += 0.0 if fluid[-1, -1, -1] else 1e-30
    iw = solver.cg(3000, 1e-9)
    assert abs(int(iw.iterations) - int(info.iterations)) <= 2
    assert rel_err(x, solver.download_x()) <= 1e-8


def test_box_keeps_what_lies_outside_the_fluid(solver):
    # decoupled cells with a right-hand side keep their solution b / c, and
    # values that a solve of the whole grid reports are still reported
    shape, levels = (96, 80, 64), 4
    print("case box outside", flush=True)
    block = ((20, 50), (20, 40), (20, 44))

    def system():
        return build(solver, shape, levels, block, 6)

    def rows(level):
        n = [e >> level for e in shape]
        return view(solver, solver.matrix_ptr(level), 4 * int(np.prod(n))).view(*n[::-1], 4)

    for precision in (jetgpu.JG_FP64, jetgpu.JG_MIXED):
        system()
        rhs(solver, shape)[60, 70, 90] = 2.5
        x, info = solve(solver, levels, precision)
        assert info.converged and abs(x[60, 70, 90] - 2.5) <= 1e-6
        for where in ("rhs", "centre", "coupling", "coarse"):
            system()
            if where == "rhs":
                rhs(solver, shape)[60, 70, 90] = float("nan")
            elif where == "centre":
                rows(0)[60, 70, 90, 0] = float("nan")
            elif where == "coupling":
                rows(0)[60, 70, 90, 1] = float("nan")
            else:
                rows(2)[15, 18, 22, 0] = float("nan")
            solver.check(jetgpu.lib().jg_solver_matrices_changed(solver.h), "matrices_changed")
            with pytest.raises(jetgpu.JgError):
                solve(solver, levels, precision)
    system()  # a centre beyond FP32 range is an error of the mixed solve only
    rows(0)[60, 70, 90, 0] = 1e300
    solver.check(jetgpu.lib().jg_solver_matrices_changed(solver.h), "matrices_changed")
    solve(solver, levels, jetgpu.JG_FP64)
    with pytest.raises(jetgpu.JgError):
        solve(solver, levels, jetgpu.JG_MIXED)


@pytest.mark.parametrize("shape,levels,block", [((128, 128, 128), 5, ((0, 128), (0, 44), (0, 128))),
                                                ((96, 128, 160), 4, ((0, 96), (0, 30), (10, 160)))])
@pytest.mark.parametrize("precision", [jetgpu.JG_FP64, jetgpu.JG_MIXED])
def test_box_flatter_than_deep(solver, shape, levels, block, precision):
    # a box with ny < nz: Jet's bound of the prolongation's k by min(ny, nz)
    # is the grid's, not the box's (with the box's, an asymmetric cycle); what
    # is left is the clamping at the box's edges inside the grid
    print(f"case box flat shape={shape} precision={precision}", flush=True)
    fluid = build(solver, shape, levels, block, 7)
    x, info = solve(solver, levels, precision)
    assert info.converged and info.rel_residual <= 1e-8
    b = rhs(solver, shape)
    b[0, 0, 0] += 0.0 if fluid[0, 0, 0] else 1e-30
    b[-1, -1, -1] += 0.0 if fluid[-1, -1, -1] else 1e-30
    whole, i2 = solve(solver, levels, precision)  # whole grid
    print("iterations", int(info.iterations), int(i2.iterations), flush=True)
    assert rel_err(x, whole) <= 1e-6
    assert int(info.iterations) <= int(i2.iterations) + 2
