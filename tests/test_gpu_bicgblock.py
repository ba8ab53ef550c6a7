"""k_bicg_block, BiCGStab with a system's whole state on chip (the default above 2048 rows with a norm-2 criterion): the
sizes and numbers of right-hand sides on both sides of every line where another instance is chosen, right-hand sides
together and one after the other, ragged 3-D blocks, transposed solves, and systems it leaves to the general kernels,
against the FP64 residual and the general kernels (PICT_CG_LOCAL_WGS selects them).

Bound: the recurrence residual ends below the tolerance; the true residual differs from it by rounding, at most a few
ulp of |A| |x| per update, taken as 16 eps ||A|| |x| row by row (as for k_cg_block)."""
import numpy as np
import pytest
import torch

from pict_amd import PISOtorch as P
from test_gpu_cgblock import walls
from test_gpu_solver import NORM2N, irregular, periodic_laplacian, to_pict

pytestmark = pytest.mark.gpu

F32, F64 = torch.float32, torch.float64


def opts(tol, maxit=500, transpose=False, zero_shortcut=0):
    o = P._solve_opts(maxit, tol, NORM2N, True, False, 0, transpose, False, False, False)
    o.zero_rhs_shortcut = zero_shortcut
    return o


def solve(A, b, tol, x0=None, **kw):
    x = torch.zeros_like(b) if x0 is None else x0.clone()
    return x, P._solve(A, b, x, opts(tol, **kw))


def skewed(shape, build=walls, shift=0.4):
    """An advection-like matrix: the Laplacian with unsymmetric values, diagonally dominant."""
    m = build(shape, shift)
    m.data = m.data * (1 + 0.3 * np.random.default_rng(5).random(m.data.shape))
    m = m.tocsr()
    m.setdiag(np.asarray(abs(m).sum(axis=1)).ravel() * 0.6)
    m.sort_indices()
    return m


def rhs(n, nr, seed, dtype):
    g = torch.Generator().manual_seed(seed)
    return (torch.rand(n * nr, generator=g, dtype=torch.float64) * 2 - 1).to(dtype).cuda()


def check_residual(m, x, b, k, tol):
    n, eps = m.shape[0], float(torch.finfo(x.dtype).eps)
    xk, bk = x[k * n:(k + 1) * n].double().cpu().numpy(), b[k * n:(k + 1) * n].double().cpu().numpy()
    r = np.linalg.norm(bk - m @ xk)
    bound = tol * np.sqrt(n) + 16 * eps * np.linalg.norm(abs(m) @ np.abs(xk))
    assert r <= bound, (k, r, bound)


def check(m, nr, dtype, name_part, monkeypatch, on_chip=True):
    A, n = to_pict(m, dtype), m.shape[0]
    b = rhs(n, nr, 3, dtype)
    b[:n] *= 1e-2  # the right-hand sides end at different iterations
    name = P.solver_kernel_name(A, nr, opts(1e-6))
    print("case", m.shape, nr, dtype, name, flush=True)
    assert name_part in name, name
    tol = 1e-12 if dtype == F64 else 1e-6
    x, infos = solve(A, b, tol)
    assert on_chip is None or all(i.onChip == on_chip for i in infos)  # which kernel solved it, not only which one was planned
    x2, _ = solve(A, b, tol)
    assert torch.equal(x, x2)
    monkeypatch.setenv("PICT_CG_LOCAL_WGS", "64")
    assert "k_bicg_block" not in P.solver_kernel_name(A, nr, opts(1e-6))
    _, ref = solve(A, b, tol)
    assert not any(i.onChip for i in ref)
    monkeypatch.delenv("PICT_CG_LOCAL_WGS")
    for k in range(nr):
        assert infos[k].converged and infos[k].isFiniteResidual and infos[k].finalResidual < tol
        assert abs(infos[k].usedIterations - ref[k].usedIterations) <= 1 + 0.05 * ref[k].usedIterations
        check_residual(m, x, b, k, tol)


# 5-entry rows: rows per thread 1, 2, 4, 8; one right-hand side, two together, three and four one after the other
@pytest.mark.parametrize("shape,rpt", [((2049, 1), 1), ((241, 17), 1), ((128, 256), 1), ((181, 182), 2), ((256, 512), 2),
                                       ((257, 513), 4), ((725, 724), 8)])
@pytest.mark.parametrize("nr", [1, 2, 3, 4])
def test_2d(shape, rpt, nr, monkeypatch):
    check(skewed(shape), nr, F32, "<float, %d, 5, %d>" % (rpt, 2 if nr == 2 else 1), monkeypatch)


@pytest.mark.parametrize("shape,rpt", [((683, 4), 2), ((97, 61), 2), ((363, 362), 4)])
@pytest.mark.parametrize("nr", [1, 2, 3])
def test_2d_fp64(shape, rpt, nr, monkeypatch):
    check(skewed(shape, periodic_laplacian), nr, F64, "<double, %d, 5, %d>" % (rpt, 2 if nr == 2 else 1), monkeypatch)


# 7-entry rows: blocks of lines that do not divide the grid; three together up to four rows per thread
@pytest.mark.parametrize("shape,rpt", [((13, 13, 13), 1), ((24, 17, 16), 1), ((57, 35, 30), 2), ((31, 59, 61), 4),
                                       ((200, 7, 90), 4), ((90, 71, 73), 8), ((110, 101, 99), 14)])
@pytest.mark.parametrize("nr", [1, 2, 3])
def test_3d(shape, rpt, nr, monkeypatch):
    together = 3 if nr == 3 and rpt <= 4 else 1
    check(skewed(shape), nr, F32, "<float, %d, 7, %d>" % (rpt, together), monkeypatch)


@pytest.mark.parametrize("shape,rpt", [((24, 17, 16), 1), ((33, 35, 40), 2), ((61, 47, 43), 4)])
@pytest.mark.parametrize("nr", [1, 3])
def test_3d_fp64(shape, rpt, nr, monkeypatch):
    together = 3 if nr == 3 and rpt <= 2 else 1
    check(skewed(shape, periodic_laplacian), nr, F64, "<double, %d, 7, %d>" % (rpt, together), monkeypatch)


# lines that leave no room for two of them in the halo are cut into strips
@pytest.mark.parametrize("shape,rpt", [((449, 70), 1), ((512, 64), 1), ((1500, 21), 1), ((512, 128), 2), ((1000, 100), 2),
                                       ((700, 400), 4), ((1000, 1000), 8)])
@pytest.mark.parametrize("nr", [1, 2])
def test_strips_2d(shape, rpt, nr, monkeypatch):
    check(skewed(shape, periodic_laplacian), nr, F32, "<float, %d, 5, %d>" % (rpt, nr), monkeypatch)


@pytest.mark.parametrize("shape,rpt", [((400, 10, 9), 1), ((1000, 9, 8), 2), ((700, 13, 15), 4), ((800, 23, 30), 8),
                                       ((512, 48, 40), 14)])
def test_strips_3d(shape, rpt, monkeypatch):
    check(skewed(shape), 3, F32, "<float, %d, 7, %d>" % (rpt, 3 if rpt <= 4 else 1), monkeypatch)


@pytest.mark.parametrize("shape,nr", [((1000, 50), 2), ((400, 10, 9), 3), ((1000, 9, 8), 3)])
def test_strips_fp64(shape, nr, monkeypatch):
    check(skewed(shape), nr, F64, "k_bicg_block<double", monkeypatch)


@pytest.mark.parametrize("dtype", [F64, F32])
def test_left_to_the_general_kernel(dtype, monkeypatch):
    """Two long lines (no interior row shows their length), columns all over the system, rows longer than the registers."""
    check(skewed((3000, 2)), 2, dtype, "k_bicg_block", monkeypatch, on_chip=dtype == F32)  # (512 and 1024 rows)
    check(skewed((3000, 4)), 2, dtype, "k_bicg_block", monkeypatch)
    check(irregular(20000, 3), 2, dtype, "", monkeypatch, on_chip=False)
    m = walls((120, 100), 0.05).tolil()
    m[0, ::1500] = -0.01  # one row of 10 entries and its mirror
    m[::1500, 0] = -0.01
    m[0, 0] = 5.0
    check(m.tocsr(), 2, dtype, "k_bicg_block", monkeypatch, on_chip=False)


@pytest.mark.parametrize("shape,nr", [((96, 64), 2), ((96, 64), 3), ((33, 20, 21), 3)])
@pytest.mark.parametrize("dtype", [F64, F32])
def test_transposed(shape, nr, dtype):
    """A transposed solve is bitwise the solve of the explicit transpose (same values in the same order)."""
    m = skewed(shape, periodic_laplacian)
    mt = m.T.tocsr()
    mt.sort_indices()
    A, At, b = to_pict(m, dtype), to_pict(mt, dtype), rhs(m.shape[0], nr, 2, dtype)
    assert "k_bicg_block" in P.solver_kernel_name(A, nr, opts(1e-6))
    xt, it = solve(A, b, 1e-6, transpose=True)
    xe, ie = solve(At, b, 1e-6)
    assert all(i.onChip for i in it + ie)
    assert [i.usedIterations for i in it] == [i.usedIterations for i in ie] and torch.equal(xt, xe)


@pytest.mark.parametrize("shape,nr", [((100, 90), 2), ((100, 90), 3), ((24, 17, 16), 3)])
def test_limits_zero_and_not_finite(shape, nr):
    m = skewed(shape)
    n = m.shape[0]
    A, b, x0 = to_pict(m, F32), rhs(n, nr, 4, F32), rhs(n, nr, 5, F32)
    assert "k_bicg_block" in P.solver_kernel_name(A, nr, opts(1e-6))
    # no iterations: the start vectors, not converged
    x, infos = solve(A, b, 1e-6, x0=x0, maxit=0)
    assert torch.equal(x, x0) and all(i.usedIterations == -1 and not i.converged for i in infos)
    # the iteration limit: the residual after it is reported
    x, infos = solve(A, b, 1e-30, maxit=3)
    for k, info in enumerate(infos):
        assert info.onChip and info.usedIterations == 2 and not info.converged and info.isFiniteResidual
        r = b[k * n:(k + 1) * n].double().cpu().numpy() - m @ x[k * n:(k + 1) * n].double().cpu().numpy()
        r = np.linalg.norm(r) / np.sqrt(n)
        assert abs(r - info.finalResidual) <= 1e-3 * r + 1e-7
    # a start that is the answer converges before the first iteration and stays; the others are solved
    xs, _ = solve(A, b, 1e-6)
    start = torch.zeros_like(b)
    start[-n:] = xs[-n:]
    x, infos = solve(A, b, 1e-5, x0=start)
    assert infos[nr - 1].usedIterations == -1 and torch.equal(x[-n:], xs[-n:])
    assert all(i.converged for i in infos) and infos[0].usedIterations >= 0
    # zero right-hand sides: the shortcut needs all of them
    x, infos = solve(A, torch.zeros_like(b), 1e-6, x0=x0, zero_shortcut=1)
    assert float(x.abs().max()) == 0.0 and all(i.converged and i.usedIterations == -1 for i in infos)
    one = b.clone()
    one[:n] = 0
    x, infos = solve(A, one, 1e-6, x0=x0, zero_shortcut=1)
    assert infos[0].converged and infos[0].usedIterations >= 0 and 0 < float(x[:n].abs().max()) < 1e-4
    # a right-hand side that is not finite ends its own solve only (an infinite one by way of the general kernel, whose
    # answers to the others differ in rounding)
    for bad in (float("nan"), float("inf")):
        bb = b.clone()
        bb[n // 2] = bad
        x, infos = solve(A, bb, 1e-6, maxit=50)
        assert not infos[0].converged and not infos[0].isFiniteResidual
        assert all(i.converged for i in infos[1:])
        check_residual(m, x, b, nr - 1, 1e-6)
        assert np.isinf(bad) or torch.equal(x[-n:], xs[-n:])
