"""The GEMM's kernel choice on the host: plans and shared launches over the range of K (no GPU).

gemm_plan and gemm_group_config are plain functions of the sizes; they are called in the built library, in a
process of their own so that a crash in them is a failed test.
"""

from __future__ import annotations

import subprocess
import sys
import textwrap

from kernelforge import build

CALLS = textwrap.dedent("""
    import ctypes, itertools, sys

    class Plan(ctypes.Structure):
        _fields_ = [(f, ctypes.c_int) for f in ("cfg", "family", "bm", "bn", "threads", "splits", "stages")]

    lib = ctypes.CDLL(sys.argv[1])
    plan = lib._ZN2kf9gemm_planEiiii
    plan.restype = Plan
    group = lib._ZN2kf17gemm_group_configEPKNS_8GemmPlanEPKiiiii
    for k, m in itertools.product((64, 128, 192, 256, 320, 2048, 5632), (5, 8, 17, 64, 200, 517, 2048)):
        for ns in ((256, 256), (64, 64, 64), (64, 8960), (4096, 4096)):
            plans = (Plan * len(ns))(*[plan(m, n, k, 256) for n in ns])
            assert all(p.splits >= 1 and (m > 16 or p.splits == 1) for p in plans), (m, ns, k)
            print(k, m, ns, group(plans, (ctypes.c_int * len(ns))(*ns), len(ns), m, k, 256), flush=True)
""")


def test_shared_launches_are_planned_for_every_k():
    run = subprocess.run([sys.executable, "-c", CALLS, str(build.LIB_PATH)], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, f"{run.returncode} after {run.stdout.splitlines()[-1:]}: {run.stderr[-500:]}"
    assert len(run.stdout.splitlines()) == 7 * 7 * 4
