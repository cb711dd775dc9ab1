"""Helper-level unit tests (the reference's UT tier, tests/train/flash_attention/ut/): the integer index
arithmetic of the kernels -- workgroup map, LDS swizzles, head-dim classes, the dK/dV query split -- lives in
a header without HIP in it, so a host compiler builds the checks and they run without a GPU."""
import os
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_index_math_host_build(tmp_path):
    src = os.path.join(ROOT, "tests", "host", "index_math_test.cpp")
    exe = str(tmp_path / "index_math_test")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-o", exe, src], check=True)
    res = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    sys.stdout.write(res.stdout)
    assert res.returncode == 0, res.stdout[-2000:]
    assert "all checks passed" in res.stdout


def _plans(tmp_path, problems):
    src, exe = os.path.join(ROOT, "tests", "host", "launch_plan.cpp"), str(tmp_path / "launch_plan")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-o", exe, src], check=True)
    text = "\n".join(" ".join(str(int(x)) for x in p) for p in problems)
    out = subprocess.run([exe], input=text, capture_output=True, text=True, check=True, timeout=60).stdout
    return [dict(zip(("kg", "kv_split", "dq_kg", "ngk", "q_split", "pipelined"), map(int, line.split()))) for line in out.splitlines()]


def test_the_gpu_tests_of_one_kernel_run_it(tmp_path):
    """The launch plan decides which kernel a shape reaches: the parity tests written for a kernel are large enough."""
    import test_gpu_parity as gpu
    rows = [(4, gpu.DQ64_BLOCKS // (4 * (Sq // 256)), Sq, Sk, 128, causal) for Sq, Sk, causal in gpu.DQ64_SHAPES]
    for row, plan in zip(rows, _plans(tmp_path, rows)):
        assert plan["dq_kg"] == 1, (row, plan)
    rows = [gpu.FULL_GRID_HEADS + (Sq, Sk, D, side == "causal") for D, Sq, Sk, side in gpu.FULL_GRIDS]
    plans = _plans(tmp_path, rows)
    for row, plan in zip(rows, plans):
        assert (plan["kg"], plan["kv_split"], plan["dq_kg"], plan["q_split"]) == (1, 1, 1, 1), (row, plan)
    assert sum(plan["ngk"] == 2 for row, plan in zip(rows, plans) if row[4] == 40) >= 3, plans


def test_the_two_key_group_tests_run_two(tmp_path):
    """The shapes written for two key groups per wave of the dK/dV kernel get them from the plan."""
    import test_key_bias_and_row_statistics as gpu
    rows = [shape + (nxt == 0,) for shape, mask, nxt, biased, keep in gpu.TWO_KEY_GROUPS]
    for row, plan in zip(rows, _plans(tmp_path, rows)):
        assert (plan["ngk"], plan["q_split"]) == (2, 1), (row, plan)
    rows = [(1, heads, D, 256, D, False) for heads, D in ((256, 64), (256, 80), (256, 128), (2, 64), (2, 80), (2, 128))]
    assert [plan["ngk"] for plan in _plans(tmp_path, rows)] == [2, 2, 2, 1, 1, 1]


def test_the_gpu_tests_of_the_pipelined_forward_run_it(tmp_path):
    import test_pipelined_forward as gpu
    cases = [(c, long) for long, some in ((0, gpu.SHORT), (1, gpu.LONG)) for c in some if c[3] in ("none", "causal", "causal tensor")]
    for tri in (0, 1):                                        # (a mask tensor is planned as if it hid nothing)
        some = [(c, long) for (c, long) in cases if (c[3] == "causal") == tri]
        for ((Sq, Sk, D, side), long), plan in zip(some, _plans(tmp_path, [gpu.heads(c[0]) + c[:3] + (tri,) for c, _ in some])):
            assert (plan["kg"], plan["kv_split"], plan["pipelined"]) == (1, 1, long), (Sq, Sk, D, side, plan)


def test_the_gpu_tests_of_launches_of_several_rounds_run_them(tmp_path):
    from test_key_group_merge import LATE_TILES, LONE_MERGES
    for whole in (True, False):
        rows = [(B if whole else B // parts, N, Sq, Sk, D, 0) for B, N, Sq, Sk, D, parts in LONE_MERGES]
        for (B, N, Sq, Sk, D, _), plan in zip(rows, _plans(tmp_path, rows)):
            assert plan["kg"] == 2 and (B * N * ((Sq + 127) // 128) > 256) == whole, (B, N, Sq, Sk, D, plan)
        rows = [(B if whole else B // parts, N, Sq, Sk, D, 0) for B, N, Sq, Sk, D, parts in LATE_TILES]
        for (B, N, Sq, Sk, D, _), plan in zip(rows, _plans(tmp_path, rows)):
            assert plan["kg"] == 1 and Sq <= 256 and Sk <= 128 and (B * N > 256) == whole, (B, N, Sq, Sk, D, plan)
