"""Gradients of static boundary velocities: one value for every cell of a face, so its gradient is the sum of the
gradients of the same velocity given per cell.  Faces that fill many workgroups, end inside one, and share a workgroup
with the opposite face, in 2-D and 3-D.

Bound: both sides compute the same terms and differ in the order of their sums only.  A cell's own sum has at most 10
terms (one rounding each, of a partial sum no larger than the sum of their magnitudes) and one more rounding follows
where the sum is stored: 11 eps times the terms' magnitudes.  Those are taken as at most 8 times the cells' sums: the
cotangents are random, so a cell's terms cancel by chance only.  The sum over the cells is held in 64 bits on both
sides; its roundings add the number of cells times the 64-bit eps.
"""
import pytest
import torch

from grad_util import OUTPUTS, create_grads
from oracle import oracle as O
from pict_amd import PISOtorch as P
from pict_amd.configs import uniform_coords

pytestmark = pytest.mark.gpu

DT = 0.05
STAGES = {
    "advection velocity": (lambda d, dt: P.SetupAdvectionVelocityGrad(d, dt, 0), ["VELOCITY_RHS"]),
    "pressure divergence": (P.SetupPressureRHSdivGrad, ["PRESSURE_RHS_DIV"]),
    "pressure right-hand side": (P.SetupPressureRHSGrad, ["PRESSURE_RHS", "PRESSURE_RHS_DIV"]),
}


def _gradients(stage, size, varying, dtype):
    dims = len(size)
    d = P.Domain(dims, torch.tensor([0.03], dtype=dtype), "walls", dtype, "cuda", passiveScalarChannels=0)
    b = d.CreateBlock(vertexCoordinates=uniform_coords(*size, dtype=dtype))
    b.CloseAllBoundaries()
    if dims == 3:
        b.MakePeriodic("z")
    gen = torch.Generator().manual_seed(1)

    def draw(t):
        return (torch.rand(t.shape, generator=gen, dtype=torch.float64) - 0.5).to(dtype=dtype, device="cuda")

    b.setVelocity(draw(b.velocity))
    walls = []
    for face, v in (("-y", 0.3), ("+y", 0.7)):
        b.CloseBoundary(face, velocity=torch.tensor([[v, -0.1, 0.2][:dims]], dtype=dtype, device="cuda"))
        walls.append(b.getBoundary(face))
        if varying:
            walls[-1].makeVelocityVarying()
    d.PrepareSolve()
    tdt = torch.tensor([DT], dtype=dtype)
    P.SetupAdvectionMatrix(d, tdt, 0)
    P.SetupAdvectionVelocity(d, tdt, 0)
    d.setVelocityResult(draw(d.velocityResult))
    d.UpdateDomainData()
    P.SetupPressureCorrection(d, tdt, 0)
    create_grads(d)
    backward, outputs = STAGES[stage]
    for o in outputs:
        OUTPUTS[o][1](d, draw(OUTPUTS[o][0](O.cpu_twin(d))))
    d.UpdateDomainData()
    backward(d, tdt)
    return [w.velocityGrad.double() for w in walls]


@pytest.mark.parametrize("stage", list(STAGES))
@pytest.mark.parametrize("size", [(7, 5), (61, 3), (300, 20), (9, 5, 6), (40, 24, 20), (33, 3, 35)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_static_wall_gradient_is_the_sum_over_cells(stage, size, dtype):
    print("case", stage, size, dtype, flush=True)
    for gs, gv in zip(_gradients(stage, size, False, dtype), _gradients(stage, size, True, dtype)):
        cells = gv.reshape(gv.shape[1], -1)
        eps = 88 * torch.finfo(dtype).eps + cells.shape[1] * torch.finfo(torch.float64).eps
        err = (gs.reshape(-1) - cells.sum(1)).abs()
        bound = eps * cells.abs().sum(1)
        print("  %.2e of %.2e" % (float(err.max()), float(bound.max())))
        assert bool((err <= bound).all()), (err, bound)
        assert float(gs.abs().max()) > 0.0
