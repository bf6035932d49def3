"""The rules of csrc/qmm_route.h (which rows a workgroup takes), through a small
host program: no device needed."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "npu880-mtk-npu-llm-runtime_amd")


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("route") / "route_caller")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-I", os.path.join(PKG, "csrc"),
                        os.path.join(ROOT, "tests", "route_caller.cpp"), "-o", exe],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr

    def ask(lines):
        out = subprocess.run([exe], input="\n".join(lines) + "\n", capture_output=True, text=True, timeout=60)
        assert out.returncode == 0, out.stderr
        got = out.stdout.splitlines()
        assert len(got) == len(lines)
        return got
    return ask


def test_rmsnorm_rows_cover_and_balance(route):
    """Every row once, and past 256 rows no XCD takes more than one row over
    its eighth."""
    Ms = [1, 15, 16, 17, 255] + list(range(256, 300)) + [511, 512, 513, 520, 560, 1000, 2047, 2048]
    for M, line in zip(Ms, route([f"rms_rows {M}" for M in Ms])):
        bad, *xcd = map(int, line.split())
        assert bad == 0 and sum(xcd) == M, (M, line)
        assert max(xcd) <= (M + 7) // 8, (M, xcd)


def test_swiglu_quads_cover_and_balance(route):
    """Every token's every quad once; the XCDs' workgroups differ by at most one
    unit of 8 tokens and one ragged unit."""
    cases = [(M, nq) for M in (1, 7, 8, 9, 15, 16, 17, 37, 65, 100, 257, 300, 513, 2048) for nq in (1, 3, 10, 14)]
    for (M, nq), line in zip(cases, route([f"quads {M} {nq}" for M, nq in cases])):
        bad, *xcd = map(int, line.split())
        assert bad == 0 and sum(xcd) == M * nq, (M, nq, line)
        assert max(xcd) - min(xcd) <= 8 + M % 8, (M, nq, xcd)
