"""k_cg_block, the CG with a system's whole state on chip (the default for one right-hand side and a norm-2 criterion):
sizes on both sides of every line where another instance or workgroup count is chosen, one workgroup and several, grids
whose lines do not fill tiles or workgroups, 3-D blocks of lines that end inside the grid, transposed solves, and
lines longer than the halo (cut into strips),
systems it leaves to the general kernels (long rows, too many foreign columns), against a direct FP64 solve and the
general kernels (PICT_CG_LOCAL_WGS selects them).

FP32 bound: the recurrence residual ends below the tolerance; the true residual differs from it by rounding, at most a
few ulp of |A| |x| per iteration-independent update, taken as 16 eps ||A|| |x| row by row."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla
import torch

from pict_amd import PISOtorch as P
from test_gpu_solver import NORM2N, irregular, kernel_name, periodic_laplacian, rhs, solve, to_pict

pytestmark = pytest.mark.gpu


def walls(shape, shift):
    """Laplacian with zero-flux walls: rows of 3 to 2 D + 1 entries."""
    n = int(np.prod(shape))
    idx = np.arange(n).reshape(shape[::-1])
    m = sp.diags([np.full(n, shift)], [0]).tolil().tocsr()
    for ax in range(len(shape)):
        a = np.take(idx, np.arange(idx.shape[ax] - 1), axis=ax).ravel()
        b = np.take(idx, np.arange(1, idx.shape[ax]), axis=ax).ravel()
        one = np.ones(a.size)
        m = m + sp.csr_matrix((np.concatenate([one, one, -one, -one]),
                               (np.concatenate([a, b, a, b]), np.concatenate([a, b, b, a]))), shape=(n, n))
    m.sort_indices()
    return m


def check(m, dtype, name_part, monkeypatch, seed=3, on_chip=True):
    A = to_pict(m, dtype)
    n = m.shape[0]
    b = rhs(n, seed, dtype)
    name = kernel_name(A)
    print("case", m.shape, dtype, name, flush=True)
    assert name_part in name, name
    tol = 1e-12 if dtype == torch.float64 else 1e-6
    x, info = solve(A, b, tol)
    assert info.converged and info.isFiniteResidual
    assert on_chip is None or info.onChip == on_chip  # which kernel solved it, not only which one was planned
    x2, info2 = solve(A, b, tol)
    # (the general FP64 kernel may put other rows in memory from run to run when lines are as long as its workgroups)
    assert info2.usedIterations == info.usedIterations and (torch.equal(x, x2) or (on_chip is None and not info.onChip))
    monkeypatch.setenv("PICT_CG_LOCAL_WGS", "64")
    xr, ir = solve(A, b, tol)
    assert not ir.onChip
    monkeypatch.delenv("PICT_CG_LOCAL_WGS")
    assert abs(info.usedIterations - ir.usedIterations) <= 2 + 0.03 * ir.usedIterations
    xn = x.double().cpu().numpy()
    r = b.double().cpu().numpy() - m @ xn
    eps = np.finfo(np.float64 if dtype == torch.float64 else np.float32).eps
    bound = tol * np.sqrt(n) + 16 * eps * np.linalg.norm(abs(m) @ np.abs(xn))
    assert np.linalg.norm(r) <= bound, (np.linalg.norm(r), bound)
    if dtype == torch.float64 and n <= 70000:
        xd = spla.spsolve(m.tocsc(), b.cpu().numpy())
        assert np.abs(xn - xd).max() <= 1e-8 * np.abs(xd).max()


# FP32 and FP64 lines: 512, 1024, 2048 (and 4096 FP32) rows on one workgroup
@pytest.mark.parametrize("shape", [(3, 1), (73, 7), (512, 1), (27, 19), (32, 32), (41, 25), (64, 32), (683, 3)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_one_workgroup(shape, dtype, monkeypatch):
    n = shape[0] * shape[1]
    check(walls(shape, 0.05), dtype, "one>" if n <= 2048 or dtype == torch.float32 else "several>", monkeypatch)


@pytest.mark.parametrize("shape", [(64, 64), (65, 63), (16, 16, 16), (15, 16, 17)])
def test_one_workgroup_1024_threads(shape, monkeypatch):
    check(walls(shape, 0.05), torch.float32, "1024, 4", monkeypatch)


# several workgroups: rows per thread 1, 2, 4, 8 (5-entry rows), ragged lines, periodic wraps
@pytest.mark.parametrize("shape,rpt", [((4097, 1), 1), ((241, 17), 1), ((128, 256), 1), ((181, 182), 2), ((256, 512), 2),
                                       ((257, 513), 4)])
@pytest.mark.parametrize("build", [walls, periodic_laplacian])
def test_several_workgroups_2d(shape, rpt, build, monkeypatch):
    if build is periodic_laplacian and min(shape) < 3:
        shape = (1366, 3)
    check(build(shape, 0.05), torch.float32, "512, %d, 5, several" % rpt, monkeypatch)


@pytest.mark.parametrize("shape", [(683, 4), (97, 61), (181, 182)])
def test_several_workgroups_2d_fp64(shape, monkeypatch):
    check(walls(shape, 0.05), torch.float64, "several", monkeypatch)


# 3-D: blocks of lines that do not divide the grid, planes larger and smaller than a workgroup
@pytest.mark.parametrize("shape,rpt", [((24, 17, 16), 1), ((57, 35, 30), 2), ((31, 59, 61), 4), ((200, 7, 90), 4),
                                       ((90, 71, 73), 8), ((110, 101, 99), 14)])
def test_several_workgroups_3d(shape, rpt, monkeypatch):
    check(walls(shape, 0.05), torch.float32, "512, %d, 7, several" % rpt, monkeypatch)


@pytest.mark.parametrize("shape", [(24, 17, 16), (33, 35, 40), (61, 47, 43)])
def test_several_workgroups_3d_fp64(shape, monkeypatch):
    check(periodic_laplacian(shape, 0.05), torch.float64, "several", monkeypatch)


# lines that leave no room for two of them in the halo (896, 1344 and 1792 rows) are cut into strips
@pytest.mark.parametrize("shape,rpt", [((400, 70), 1), ((449, 70), 1), ((512, 64), 1), ((1500, 21), 1), ((512, 128), 2),
                                       ((1000, 100), 2), ((640, 300), 4), ((700, 300), 4), ((700, 400), 4),
                                       ((890, 700), 8), ((897, 700), 8), ((1000, 1000), 8), ((1024, 1024), 8)])
@pytest.mark.parametrize("build", [walls, periodic_laplacian])
def test_strips_2d(shape, rpt, build, monkeypatch):
    if shape[0] * shape[1] > 500000 and build is periodic_laplacian and shape[0] != 1000:
        pytest.skip("large: once")
    check(build(shape, 0.05), torch.float32, "512, %d, 5, several" % rpt, monkeypatch)


@pytest.mark.parametrize("shape", [(1000, 50), (1000, 300)])
def test_strips_2d_fp64(shape, monkeypatch):
    check(periodic_laplacian(shape, 0.05), torch.float64, "several", monkeypatch)


@pytest.mark.parametrize("shape,rpt", [((400, 10, 9), 1), ((1000, 9, 8), 2), ((700, 13, 15), 4), ((800, 23, 30), 8),
                                       ((512, 48, 40), 14)])
def test_strips_3d(shape, rpt, monkeypatch):
    check(walls(shape, 0.05), torch.float32, "512, %d, 7, several" % rpt, monkeypatch)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_blocks_of_different_lines(dtype, monkeypatch):
    """A domain of blocks with lines of different lengths: whichever the mapping follows, the answer is right."""
    for shapes in (((600, 40), (90, 100)), ((90, 100), (600, 40)), ((30, 20, 20), (600, 5, 4)), ((600, 5, 4), (30, 20, 20))):
        m = sp.block_diag([walls(s, 0.05) for s in shapes]).tocsr()
        m.sort_indices()
        check(m, dtype, "several", monkeypatch, on_chip=None)


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_left_to_the_general_kernel(dtype, monkeypatch):
    """Two long lines (no interior row shows their length), columns all over the system, and rows longer than the
    registers: the general kernel solves them; on one workgroup long rows are read from memory."""
    check(walls((3000, 2), 0.05), dtype, "several", monkeypatch, on_chip=dtype == torch.float32)  # (512 and 1024 rows)
    check(walls((3000, 4), 0.05), dtype, "several", monkeypatch)
    check(irregular(20000, 3), dtype, "", monkeypatch, on_chip=False)
    n = 12000
    m = walls((120, 100), 0.05).tolil()
    m[0, ::1500] = -0.01  # one row of 10 entries and its mirror
    m[::1500, 0] = -0.01
    m[0, 0] = 5.0
    check(m.tocsr(), dtype, "several", monkeypatch, on_chip=False)
    m = walls((30, 30), 0.05).tolil()
    m[0, ::90] = -0.01
    m[::90, 0] = -0.01
    m[0, 0] = 5.0
    check(m.tocsr(), dtype, "one", monkeypatch)


@pytest.mark.parametrize("shape", [(30, 33), (96, 64), (33, 20, 21)])
def test_transposed(shape):
    """A transposed solve is bitwise the solve of the explicit transpose (same values in the same order)."""
    m = periodic_laplacian(shape, 0.3)
    m.data = m.data * (1 + 0.1 * np.random.default_rng(5).random(m.data.shape))
    mt = m.T.tocsr()
    mt.sort_indices()
    for dtype in (torch.float64, torch.float32):
        A, At, b = to_pict(m, dtype), to_pict(mt, dtype), rhs(m.shape[0], 2, dtype)
        assert "k_cg_block" in kernel_name(A)
        xt, it = solve(A, b, 1e-6, transpose=True, maxit=200)
        xe, ie = solve(At, b, 1e-6, maxit=200)
        assert it.onChip and ie.onChip
        assert it.usedIterations == ie.usedIterations and torch.equal(xt, xe)


@pytest.mark.parametrize("shape", [(20, 20), (100, 90)])
def test_limits_zero_and_not_finite(shape):
    m = walls(shape, 0.1)
    n = m.shape[0]
    A = to_pict(m, torch.float32)
    b = rhs(n, 4, torch.float32)
    x0 = rhs(n, 5, torch.float32)
    # no iterations: the start vector, not converged
    x, info = solve(A, b, 1e-6, maxit=0, x0=x0)
    assert torch.equal(x, x0) and info.usedIterations == -1 and not info.converged
    # the iteration limit: the residual after it is reported
    x, info = solve(A, b, 1e-30, maxit=7)
    assert info.onChip and info.usedIterations == 6 and not info.converged and info.isFiniteResidual
    r = np.linalg.norm(b.double().cpu().numpy() - m @ x.double().cpu().numpy()) / np.sqrt(n)
    assert abs(r - info.finalResidual) <= 1e-4 * r
    # the zero right-hand-side shortcut
    o = P._solve_opts(100, 1e-6, NORM2N, False, False, 0, False, False, False, False)
    o.zero_rhs_shortcut = 1
    x = x0.clone()
    infos = P._solve(A, torch.zeros_like(b), x, o)
    assert infos[0].converged and infos[0].usedIterations == -1 and float(x.abs().max()) == 0.0
    # a right-hand side that is not finite ends the solve without an answer, as in the general kernels
    for bad in (float("nan"), float("inf")):
        bb = b.clone()
        bb[n // 2] = bad
        _, info = solve(A, bb, 1e-6, maxit=50)
        assert not info.converged and not info.isFiniteResidual
