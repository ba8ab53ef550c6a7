"""bench.py's roofline entry: a kernel that keeps its system on chip is not held against bytes that it does not move."""
import bench


def test_entries():
    n, nnz = 65536, 5 * 65536
    once, its = bench.solver_bytes_once(n, nnz, 1, 4), 110
    streamed = bench.solver_bytes("CG", n, nnz, 1, 4, [its])
    assert once == nnz * 8 + (n + 1) * 4 + 3 * n * 4
    for name in ("pict::k_cg_block<float, 512, 2, 5, several>", "pict::k_bicg_block<float, 2, 5, 2>",
                 "pict::k_cg_block_jobs<float, 5>"):
        r = bench.solver_roofline(name, streamed, once, 0.23, its, None, None)
        assert r["bound"] == "latency" and r["bytes_per_launch"] == once and r["frac"] < 0.01
        assert abs(r["us_per_iteration"] - 230.0 / its) < 1e-9
    r = bench.solver_roofline("pict::k_cg1<float, 1, true>", streamed, once, 0.23, its, None, None)
    assert r["bound"] == "hbm" and r["bytes_per_launch"] == streamed and "us_per_iteration" not in r
