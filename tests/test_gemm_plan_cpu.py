"""The GEMM's kernel choice on the host: plans and shared launches over the range of K, plans within a limit
on the partials (no GPU).

gemm_plan, gemm_plan_within and gemm_group_config are plain functions of the sizes; they are called in the
built library, in a process of their own so that a crash in them is a failed test.
"""

from __future__ import annotations

import subprocess
import sys
import textwrap

from kernelforge import build

HEAD = textwrap.dedent("""
    import ctypes, itertools, sys

    class Plan(ctypes.Structure):
        _fields_ = [(f, ctypes.c_int) for f in ("cfg", "bm", "bn", "threads", "splits", "stages")]

    lib = ctypes.CDLL(sys.argv[1])
    plan = lib._ZN2kf9gemm_planEiiii
    plan.restype = Plan
""")

GROUPS = HEAD + textwrap.dedent("""
    group = lib._ZN2kf17gemm_group_configEPKNS_8GemmPlanEPKiiiii
    for k, m in itertools.product((64, 128, 192, 256, 320, 2048, 5632), (5, 8, 17, 64, 200, 517, 2048)):
        for ns in ((256, 256), (64, 64, 64), (64, 8960), (4096, 4096)):
            plans = (Plan * len(ns))(*[plan(m, n, k, 256) for n in ns])
            assert all(p.splits >= 1 and (m > 16 or p.splits == 1) for p in plans), (m, ns, k)
            print(k, m, ns, group(plans, (ctypes.c_int * len(ns))(*ns), len(ns), m, k, 256), flush=True)
""")

WITHIN = HEAD + textwrap.dedent("""
    within = lib._ZN2kf16gemm_plan_withinEiiiim
    within.restype = Plan
    limit, over = 32 << 20, 0
    size = lambda p, m, n: p.splits * m * n * 4 if p.splits > 1 else 0
    for m, n, k in itertools.product((17, 64, 200, 512, 1024, 1536, 2048, 4096), (64, 1024, 1536, 2560, 8192),
                                     (64, 2048, 8192, 16384, 32768, 65536, 131072)):
        free, held = plan(m, n, k, 256), within(m, n, k, 256, ctypes.c_size_t(limit))
        assert size(held, m, n) <= limit and held.splits >= 1, (m, n, k, held.splits)
        if size(free, m, n) <= limit:
            assert bytes(free) == bytes(held), (m, n, k)
        else:
            over += 1
        print(m, n, k, free.splits, held.splits, flush=True)
    assert over
""")

HUGE = HEAD + textwrap.dedent("""
    for m, n, k in itertools.product((2 ** 26, 2 ** 30), (2 ** 20, 2 ** 30), (64, 128, 192, 4096)):
        p = plan(m, n, k, 256)
        assert (-(-m // p.bm) * -(-n // p.bn) * p.splits + 8) * p.threads > 2 ** 31 - 1, (m, n, k)
        print(m, n, k, flush=True)
""")


def _run(calls: str) -> list[str]:
    run = subprocess.run([sys.executable, "-c", calls, str(build.LIB_PATH)], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, f"{run.returncode} after {run.stdout.splitlines()[-1:]}: {run.stderr[-500:]}"
    return run.stdout.splitlines()


def test_shared_launches_are_planned_for_every_k():
    assert len(_run(GROUPS)) == 7 * 7 * 4


def test_a_limit_on_the_partials_always_has_a_plan():
    """The limit is that of the entry point that allocates nothing: it takes every problem, with the plan of
    the workspace entry point wherever that one fits."""
    assert len(_run(WITHIN)) == 8 * 5 * 7


def test_a_problem_past_every_grid_limit_has_a_plan_that_is_past_its_own():
    """The entry points refuse such a plan; a tile deeper than K is none."""
    assert len(_run(HUGE)) == 2 * 2 * 4
