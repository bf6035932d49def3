"""The rules of csrc/qmm_route.h (which rows a workgroup takes, which kernel a GEMM
takes), through a small host program: no device needed."""
import os
import subprocess

import pytest

from oracle import TYPE_Q4_K, TYPE_Q5_K, TYPE_Q6_K
from test_gpu_wave_slabs import PREFILL

FORMAT = {TYPE_Q4_K: 4, TYPE_Q5_K: 5, TYPE_Q6_K: 6}
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


def _prefill(route, cases):
    return route([f"prefill {FORMAT[t]} {K} {M} 256 {len(rows)} {' '.join(map(str, rows))}" for t, rows, K, M in cases])


def test_prefill_kernels_of_the_gpu_cases(route):
    """Each case of the wave-slab GPU tests takes the kernel it is there for."""
    for kernel, cases in PREFILL.items():
        assert _prefill(route, [c[:4] for c in cases]) == [kernel] * len(cases), kernel


def test_prefill_q6k_256_tokens_only_where_faster(route):
    """The 32 x 256 decoded slabs' longer start: in one round beside 2 to 3 of the
    16 x 128 slabs per CU these were faster over short K (5000 x 512 at M = 192
    6.2 against 7.2 us) and where half of 256 tokens are missing over long K."""
    few = [([5000], 512, 192), ([2560], 512, 400), ([6144], 2560, 160), ([4096], 4096, 257), ([2560], 2560, 512),
           ([5000], 9728, 160)]
    assert set(_prefill(route, [(TYPE_Q6_K, *c) for c in few])) == {"D"}
    rounds = [([6144], 512, 1100), ([14336], 512, 400), ([4096], 1024, 1024)]
    assert "E" not in _prefill(route, [(TYPE_Q6_K, *c) for c in rounds])
    many = [([2560], 9728, 512), ([4096], 4096, 512), ([4096], 512, 512), ([6144], 9728, 256)]
    assert set(_prefill(route, [(TYPE_Q6_K, *c) for c in many])) == {"E"}
