"""Host logic under the address and undefined-behaviour sanitizers (CPU).

Builds two native checks with g++ -fsanitize=address,undefined and runs them:
  - tests/native/plan_check.cpp over aegean-tge_amd/host/plan.cpp: random
    step plans (decode and block-prefill work lists cover every page once,
    split slots and reduction records agree), rejected descriptions, and
    staged uploads that survive injected allocation failures;
  - tests/native/driver_host_check.cpp over aegean-tge_amd/host/qwen2_kv.cpp
    with a stand-in for the device entry points: transactional begin under
    injected plan and copy failures, exact token-by-token prefix matching,
    and a random flow whose attaches are checked against page contents.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
FLAGS = ["-std=c++20", "-O1", "-g", "-fsanitize=address,undefined",
         "-fno-sanitize-recover=all", "-Wall", "-Wextra", "-Werror",
         "-I" + os.path.join(ROOT, "include")]


def build_and_run(tmp_path, name, sources, runs=((),), flags=FLAGS):
    if not shutil.which("g++"):
        pytest.skip("g++ not available")
    exe = str(tmp_path / name)
    cmd = ["g++", *flags, *[os.path.join(ROOT, s) for s in sources], "-o", exe]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-4000:]
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:abort_on_error=0",
               UBSAN_OPTIONS="print_stacktrace=1")
    out = ""
    for args in runs:
        r = subprocess.run([exe, *map(str, args)], capture_output=True, text=True, timeout=300, env=env)
        assert r.returncode == 0, (r.stdout + r.stderr)[-4000:]
        out += r.stdout
    return out


def test_planner_under_sanitizers(tmp_path):
    out = build_and_run(tmp_path, "plan_check",
                        ["aegean-tge_amd/host/plan.cpp", "tests/native/plan_check.cpp"])
    assert "plan_check ok" in out


def test_driver_bookkeeping_under_sanitizers(tmp_path):
    out = build_and_run(tmp_path, "driver_host_check",
                        ["aegean-tge_amd/host/qwen2_kv.cpp", "tests/native/driver_host_check.cpp"])
    assert "driver_host_check ok" in out


def test_plans_of_the_gpu_cases(tmp_path):
    """The GPU tests' launches are what they are named for."""
    from _paged import PAGE_APPEND_STEP, PAGE_APPENDS, PREFILL_PLANS, ROW_APPENDS
    import tge_kv as tk
    runs = [(qh, kvh, hd, int(fmt == tk.KV_I8), ctx, n) for qh, kvh, hd, fmt, ctx, n, _, _ in PREFILL_PLANS.values()]
    steps = [x for pair in zip(*PAGE_APPEND_STEP) for x in pair]
    runs += [(2 * kvh, kvh, hd, int(fmt == tk.KV_I8), *steps) for fmt, _, kvh, hd in PAGE_APPENDS + ROW_APPENDS]
    out = build_and_run(tmp_path, "plan_check", ["aegean-tge_amd/host/plan.cpp", "tests/native/plan_check.cpp"], runs)
    plans = [dict(zip(line.split()[::2], map(int, line.split()[1::2]))) for line in out.splitlines()]
    for (name, case), p in zip(PREFILL_PLANS.items(), plans):
        kind = "whole" if p["parts"] == 0 else "cut" if p["parts"] == p["items"] else "mix"
        assert (kind, p["tile_rows"]) == case[6:], (name, p)
    for case, p in zip(PAGE_APPENDS + ROW_APPENDS, plans[len(PREFILL_PLANS):]):
        assert (p["append_pages"] > 0) == (case in PAGE_APPENDS), case


def test_append_by_page_where_it_gains(tmp_path):
    """Steps at which the row kernel measured faster than the page kernel
    store row by row (KV heads, head_dim, int8, rows), those at which the
    page kernel did store by page."""
    by_row = [(2, 256, 1, 2048), (1, 128, 1, 16384), (1, 128, 1, 32768), (4, 256, 1, 1024), (8, 256, 1, 512),
              (4, 128, 1, 3072), (4, 128, 0, 1100), (4, 128, 0, 1500), (2, 128, 0, 2600), (1, 128, 0, 6000)]
    by_page = [(8, 256, 1, 1024), (8, 128, 1, 2048), (4, 128, 1, 8192), (4, 256, 1, 2048), (2, 256, 1, 6144),
               (8, 256, 0, 257), (8, 128, 0, 513), (4, 256, 0, 515), (4, 128, 0, 2048), (2, 128, 0, 4097),
               (1, 128, 0, 8200), (2, 256, 0, 2048), (1, 256, 0, 4100)]
    out = build_and_run(tmp_path, "plan_check", ["aegean-tge_amd/host/plan.cpp", "tests/native/plan_check.cpp"],
                        [(kvh, kvh, hd, i8, 0, n) for kvh, hd, i8, n in by_row + by_page])
    for case, line in zip(by_row + by_page, out.splitlines()):
        p = dict(zip(line.split()[::2], map(int, line.split()[1::2])))
        assert (p["append_pages"] > 0) == (case in by_page), case


def test_prefill_planning_time(tmp_path):
    """A step that only stores plans its prefill too: for large steps that
    takes a third to three quarters of what the step's own records take (a
    comparison that plays every launch through took 1.8 to 4 times as long
    as they did)."""
    runs = [(14, 2, 64, 0, 0, 20000), (28, 4, 128, 1, 0, 20000), (14, 2, 64, 0, 0, 4096)]
    out = build_and_run(tmp_path, "plan_check", ["aegean-tge_amd/host/plan.cpp", "tests/native/plan_check.cpp"], runs,
                        flags=["-std=c++20", "-O2", "-I" + os.path.join(ROOT, "include")])
    for case, line in zip(runs, out.splitlines()):
        p = dict(zip(line.split()[::2], map(int, line.split()[1::2])))
        assert p["prefill_ns"] < 1.5 * p["step_ns"], (case, p)
