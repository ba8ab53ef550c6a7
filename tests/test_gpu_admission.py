"""Admission of the on-chip solvers' grids (block_admit): a grid that does not become resident as a whole leaves the
system to the general kernel, so solves on concurrent streams end with an answer.

- Declined from the host (PICT_SOLVER_ADMIT_POLLS=0): bitwise the general kernel's answer.
- Wait limits of a few polls: workgroup 0's admission races with the others' refusals; bitwise one answer or the other.
- Threads with a stream each, systems whose grids need more than half of the compute units: the same.
- Cooperative and ordinary launches of the on-chip kernels and of the general ones: bitwise the same."""
import threading

import pytest
import torch

from pict_amd import PISOtorch as P
from test_gpu_bicgblock import skewed
from test_gpu_cgblock import walls
from test_gpu_solver import NORM2N, to_pict

pytestmark = pytest.mark.gpu

F32, F64 = torch.float32, torch.float64
# (grid, rows per thread): CG and BiCGStab on several workgroups, FP32 and FP64, up to one workgroup per compute unit
CASES = [((128, 96), F32, False), ((97, 61), F64, False), ((57, 35, 30), F32, False), ((110, 101, 99), F32, False),
         ((128, 96), F32, True), ((97, 61), F64, True), ((57, 35, 30), F32, True), ((110, 101, 99), F32, True)]


def system(shape, dtype, bicg):
    m = skewed(shape) if bicg else walls(shape, 0.05)
    nr = len(shape) if bicg else 1
    g = torch.Generator().manual_seed(3)
    b = (torch.rand(m.shape[0] * nr, generator=g, dtype=torch.float64) * 2 - 1).to(dtype).cuda()
    return to_pict(m, dtype), b


def solve(A, b, bicg):
    x = torch.zeros_like(b)
    infos = P.SolveLinear(A, b, x, 2000, 1e-10 if b.dtype == F64 else 1e-6, NORM2N, bicg, False, 0, False, False, False,
                          False)
    assert all(i.converged and i.isFiniteResidual for i in infos)
    assert len({i.onChip for i in infos}) == 1
    return x, infos[0].onChip


def both(A, b, bicg, monkeypatch):
    """The answers of the on-chip and of the general kernel."""
    x, on_chip = solve(A, b, bicg)
    assert on_chip
    monkeypatch.setenv("PICT_CG_LOCAL_WGS", "64")
    y, on_chip = solve(A, b, bicg)
    monkeypatch.delenv("PICT_CG_LOCAL_WGS")
    assert not on_chip
    return x, y


@pytest.mark.parametrize("shape,dtype,bicg", CASES)
def test_declined_grids_leave_the_system_to_the_general_kernel(shape, dtype, bicg, monkeypatch):
    print("case", shape, dtype, bicg, flush=True)
    A, b = system(shape, dtype, bicg)
    x, y = both(A, b, bicg, monkeypatch)
    monkeypatch.setenv("PICT_SOLVER_ADMIT_POLLS", "0")
    z, on_chip = solve(A, b, bicg)
    assert not on_chip and torch.equal(z, y)
    monkeypatch.delenv("PICT_SOLVER_ADMIT_POLLS")
    z, on_chip = solve(A, b, bicg)
    assert on_chip and torch.equal(z, x)


@pytest.mark.parametrize("shape,dtype,bicg", CASES)
def test_few_polls(shape, dtype, bicg, monkeypatch):
    print("case", shape, dtype, bicg, flush=True)
    A, b = system(shape, dtype, bicg)
    x, y = both(A, b, bicg, monkeypatch)
    seen = []
    for polls in (1, 2, 4, 8, 16, 32):
        monkeypatch.setenv("PICT_SOLVER_ADMIT_POLLS", str(polls))
        for _ in range(4):
            z, on_chip = solve(A, b, bicg)
            assert torch.equal(z, x if on_chip else y), (polls, on_chip)
            seen.append(on_chip)
    print(" on chip", sum(seen), "of", len(seen), flush=True)


@pytest.mark.parametrize("shape,dtype", [((110, 101, 99), F32), ((256, 256), F32), ((320, 256), F64)])
def test_concurrent_streams(shape, dtype, monkeypatch):
    print("case", shape, dtype, flush=True)
    systems = [(bicg,) + system(shape, dtype, bicg) for bicg in (False, True)]
    answers = [both(A, b, bicg, monkeypatch) for bicg, A, b in systems]
    torch.cuda.synchronize()
    failures, counts = [], []

    def work(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for i in range(8):
                    j = (k + i) % 2
                    bicg, A, b = systems[j]
                    z, on_chip = solve(A, b, bicg)
                    counts.append(on_chip)
                    if not torch.equal(z, answers[j][0 if on_chip else 1]):
                        failures.append((k, i, on_chip))
        except Exception as e:  # noqa: BLE001
            failures.append((k, repr(e)))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    print(" on chip", sum(counts), "of", len(counts), flush=True)
    assert not failures and len(counts) == 24


@pytest.mark.parametrize("shape,dtype,bicg", CASES)
@pytest.mark.parametrize("general", [False, True])
def test_launch_kinds(shape, dtype, bicg, general, monkeypatch):
    print("case", shape, dtype, bicg, general, flush=True)
    A, b = system(shape, dtype, bicg)
    if general:
        monkeypatch.setenv("PICT_CG_LOCAL_WGS", "64")
    out = []
    for plain in ("1", "0"):
        monkeypatch.setenv("PICT_SOLVER_PLAIN_LAUNCH", plain)
        x, on_chip = solve(A, b, bicg)
        assert on_chip == (not general)
        out.append(x)
    assert torch.equal(out[0], out[1])


@pytest.mark.parametrize("shape,dtype,bicg", CASES)
def test_a_wait_that_runs_out_ends_the_solve(shape, dtype, bicg, monkeypatch):
    """With no polls allowed after admission the first wait that is not over at once ends its workgroup and then the
    others: an error, no second wait, and the next solve is not affected."""
    print("case", shape, dtype, bicg, flush=True)
    A, b = system(shape, dtype, bicg)
    x, _ = both(A, b, bicg, monkeypatch)
    monkeypatch.setenv("PICT_SOLVER_SPIN_LIMIT", "0")
    with pytest.raises(Exception, match="spin limit"):
        solve(A, b, bicg)
    monkeypatch.delenv("PICT_SOLVER_SPIN_LIMIT")
    z, on_chip = solve(A, b, bicg)
    assert on_chip and torch.equal(z, x)
