"""Partial sums travel between the workgroups of the on-chip solvers whole: a system whose sums are exact in FP64 as long
as no bit of a workgroup's partial sum is dropped.

One workgroup holds all nonzero entries, 2^26 and a few ones, whose squares sum to integers with all 53 bits in use
(every order of the additions is exact); the matrix is diagonal (the grid's pattern, its other values 0) with entries 3
and 1 on equal halves, so alpha = (r, r) / (r, A r) = 1/2 and the next residual is r / 2, up to sign.  The reported
residual norm is then the rounded square root of a known number; without the lowest two bits of the sums it would be two
units in the last place less."""
import math

import numpy as np
import pytest
import torch

from pict_amd import PISOtorch as P
from test_gpu_cgblock import walls
from test_gpu_solver import to_pict

pytestmark = pytest.mark.gpu

F32, F64 = torch.float32, torch.float64
NORM2 = P.ConvergenceCriterion.NORM2


def system(shape, dtype, nr):
    m = walls(shape, 0.05).tocsr()
    m.data[:] = 0.0
    n = m.shape[0]
    diag = np.ones(n)
    diag[:8:2] = 3.0
    rows = np.repeat(np.arange(n), np.diff(m.indptr))
    m.data[m.indices == rows] = diag
    b = torch.zeros(nr, n, dtype=torch.float64)
    b[:, :8] = 1.0
    b[:, :2] = 2.0 ** 26
    return to_pict(m, dtype), b.reshape(-1).to(dtype).cuda()


S = 2 ** 52 + 3  # of either half


@pytest.mark.parametrize("shape,dtype", [((128, 96), F32), ((256, 256), F32), ((257, 513), F32), ((640, 500), F32),
                                         ((24, 17, 16), F32), ((57, 35, 30), F32), ((31, 59, 61), F32),
                                         ((90, 71, 73), F32), ((110, 101, 99), F32), ((97, 61), F64), ((363, 362), F64),
                                         ((24, 17, 16), F64), ((33, 35, 40), F64), ((61, 47, 43), F64)])
def test_cg(shape, dtype):
    print("case", shape, dtype, flush=True)
    A, b = system(shape, dtype, 1)
    x = torch.zeros_like(b)
    info = P.SolveLinear(A, b, x, 1, 1e-30, NORM2, False, False, 0, False, False, False, False)[0]
    assert info.onChip and info.usedIterations == 0
    assert info.finalResidual == math.sqrt(S / 2)
    assert torch.equal(x, b / 2)


@pytest.mark.parametrize("shape,dtype,nr", [((128, 96), F32, 2), ((256, 256), F32, 1), ((256, 256), F32, 2),
                                            ((257, 513), F32, 2), ((640, 500), F32, 2), ((24, 17, 16), F32, 3),
                                            ((57, 35, 30), F32, 3), ((57, 35, 30), F32, 4), ((31, 59, 61), F32, 3),
                                            ((90, 71, 73), F32, 3), ((110, 101, 99), F32, 3), ((97, 61), F64, 2),
                                            ((363, 362), F64, 2), ((24, 17, 16), F64, 3), ((33, 35, 40), F64, 3)])
def test_bicgstab(shape, dtype, nr):
    print("case", shape, dtype, nr, flush=True)
    A, b = system(shape, dtype, nr)

    def solve(tol):
        x = torch.zeros_like(b)
        infos = P.SolveLinear(A, b, x, 10, tol, NORM2, True, False, 0, False, False, False, False)
        assert all(i.onChip and i.converged for i in infos)
        return x, infos

    # converged at the start, and at the half step of the first iteration
    x, infos = solve(1e30)
    assert all(i.finalResidual == math.sqrt(2 * S) for i in infos) and float(x.abs().max()) == 0.0
    x, infos = solve(math.sqrt(S))
    assert all(i.finalResidual == math.sqrt(S / 2) and i.usedIterations == 0 for i in infos)
    assert torch.equal(x, b / 2)
