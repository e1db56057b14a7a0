"""The launch planners (blog_amd/csrc/qlin_plan.hpp), on the CPU: tests/plan_check.cpp (LDS arithmetic, choices of
kernels) and tests/plan_route.cpp (the kernel of a product) are built with g++ against the same header the
kernels' launchers include, and run."""
import os
import subprocess

import test_gpu_parity as parity

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_planners_fit_lds_up_to_the_edge(tmp_path):
    exe = tmp_path / "plan_check"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{os.path.join(ROOT, 'blog_amd', 'csrc')}",
                    os.path.join(ROOT, "tests", "plan_check.cpp"), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.startswith("ok")


def test_parity_cases_take_the_kernels_they_name(tmp_path):
    """Every tile kind of every format, store and SwiGLU, has a case in the parity tests, and the cases written for
    one kernel still reach it: a cost measured again must not move them elsewhere unnoticed."""
    exe = tmp_path / "plan_route"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", f"-I{os.path.join(ROOT, 'blog_amd', 'csrc')}",
                    os.path.join(ROOT, "tests", "plan_route.cpp"), "-o", str(exe)], check=True)
    want = []
    for t, n, k, m, store, swiglu in parity.BLOCK_ROWS:
        want += [((t, n, k, m, 0), (store,)), ((t, n, k, m, 1), (swiglu,))]
    want += [((*c, 0), ("super", "super small")) for c in parity.F32_GEMM_SCALES + parity.F32_GEMM_ADD]
    want += [((t, n, 1024, m, 0), ("1x1",) if n == 300 else ("mid", "large")) for t, n, m in parity.WIDE_ROWS]
    want += [((t, n, k, m, 0), ("super" if m > 100 else "super small",)) for t, n, k, m in
             [(parity.Q6_K, 8192, 2048, 512), (parity.Q6_K, 8192, 2048, 80)]]
    # the MoE FFN calls whose shared down projection is a GEMM
    want += [((parity.Q4_K, 512, 512, 70, 0), ("super small",)), ((parity.Q8_0, 2304, 96, 300, 0), ("mid",))]
    out = subprocess.run([str(exe)], input="".join(" ".join(map(str, c)) + "\n" for c, _ in want), text=True,
                         capture_output=True, check=True).stdout.split("\n")
    bad = [(c, w, got) for (c, w), got in zip(want, out) if got not in w]
    assert not bad, bad
    kinds = {(c[0], c[4], got) for (c, _), got in zip(want, out)}
    for t in (parity.Q4_0, parity.Q5_0, parity.Q8_0):
        assert {k for tt, sw, k in kinds if (tt, sw) == (t, 0)} == {"1x1", "2x1", "2x2", "2x3", "2x4", "mid", "large"}, t
        assert {k for tt, sw, k in kinds if (tt, sw) == (t, 1)} == {"2x1", "2x2", "2x3", "2x4", "mid", "large"}, t
    assert {k for tt, sw, k in kinds if (tt, sw) == (parity.Q6_K, 0)} >= {"1x1", "1x2", "2x1", "2x2", "2x3"}
    assert {k for tt, sw, k in kinds if (tt, sw) == (parity.Q6_K, 1)} == {"2x1", "2x2", "2x3"}
