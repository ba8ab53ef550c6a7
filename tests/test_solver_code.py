"""Properties of the solver kernels' machine code that no run can show: orderings that hold on a GPU most of the time
without the wait that guarantees them.  The gfx950 code of the built library is disassembled; no GPU is needed."""
import os
import re
import shutil
import subprocess

import pytest

from pict_amd import build

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
pytestmark = pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")


@pytest.fixture(scope="module")
def code_objects(tmp_path_factory):
    if not os.path.exists(build.LIB):
        build.build()
    d = tmp_path_factory.mktemp("code")
    shutil.copy(build.LIB, d / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=d, check=True, capture_output=True)
    return [str(f) for f in sorted(d.iterdir()) if "gfx950" in f.name]


def instructions(files, symbol):
    for f in files:
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--disassemble-symbols=" + symbol, f],
                              check=True, capture_output=True, text=True).stdout
        if symbol in text:
            return [x.strip().split("//")[0].strip() for x in text.split(symbol + ">:")[1].splitlines() if x.strip()]
    raise AssertionError("no kernel " + symbol)


# the FP32 instances on several workgroups: rows per thread, row length, halo rows per thread, large
@pytest.mark.parametrize("rpt,nz,hpt,big", [(1, 5, 2, 0), (2, 5, 2, 0), (4, 5, 3, 0), (8, 5, 4, 0), (1, 7, 3, 0),
                                            (2, 7, 4, 0), (4, 7, 6, 0), (8, 7, 9, 0), (14, 7, 12, 1)])
def test_cg_waits_for_the_halo_marks_before_its_first_sums(code_objects, rpt, nz, hpt, big):
    """A workgroup marks the tiles of rows that it reads of others; their owners look at the marks once, after the first
    totals.  So every wave waits for its stores (vmcnt 0) behind its last store of the set-up, the publication of its
    rows, and before the barrier at which wave 0 posts the workgroup's first sums."""
    sym = "_ZN4pict10k_cg_blockIfLi512ELi%dELi%dELi%dELb%dELb0EEEvNS_9SolveArgsIT_EE" % (rpt, nz, hpt, big)
    ins = instructions(code_objects, sym)
    out = [i for i, x in enumerate(ins) if re.match(r"global_store_dwordx2 .*sc1", x)]
    assert any(re.match(r"global_store_dword .*sc1", x) for x in ins[:out[0]])  # the marks
    # rows are published one per thread and row, then the first pair of sums is posted, behind a reduction across lanes
    post = next(i for i, j in zip(out[1:], out) if any("_dpp" in x for x in ins[j:i]))
    rows = max(i for i in out if i < post)
    barrier = max(i for i in range(rows, post) if ins[i].startswith("s_barrier"))
    assert any(re.match(r"s_waitcnt .*vmcnt\(0\)", x) for x in ins[rows:barrier])
