"""The rules of csrc/qmm_route.h (which rows a workgroup takes, which kernel a GEMM
takes), through a small host program: no device needed."""
import os
import subprocess

import pytest

from oracle import TYPE_Q4_K, TYPE_Q5_K, TYPE_Q6_K
from test_gpu_wave_slabs import EXTREME, PREFILL, TALL

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


def test_swiglu_blocks_cover_and_balance(route):
    """Every token's every block once, no workgroup without a block but for
    missing tokens; the XCDs' waves differ by at most two runs of 8 workgroups
    (one run, and one of a ragged token group)."""
    cases = [(M, nb) for M in (1, 7, 8, 9, 15, 16, 17, 37, 65, 100, 257, 300, 513, 2048)
             for nb in (1, 2, 3, 4, 5, 6, 7, 9, 10, 38, 39, 56)] + [(12000, 4095)]  # (units past 2^32 / blocks)
    for (M, nb), line in zip(cases, route([f"blocks {M} {nb}" for M, nb in cases])):
        bad, *xcd = map(int, line.split())
        assert bad == 0 and sum(xcd) == M * nb, (M, nb, line)
        assert max(xcd) - min(xcd) <= 64, (M, nb, xcd)


def _prefill(route, cases):
    return route([f"prefill {FORMAT[t]} {K} {M} 256 {len(rows)} {' '.join(map(str, rows))}" for t, rows, K, M in cases])


def test_prefill_kernels_of_the_gpu_cases(route):
    """Each case of the wave-slab GPU tests takes the kernel it is there for."""
    for kernel, cases in PREFILL.items():
        assert _prefill(route, [c[:4] for c in cases]) == [kernel] * len(cases), kernel
    assert _prefill(route, [(t, [n], K, M) for t, n, K, M in EXTREME if M > 64]) == ["A", "C", "C"]
    assert _tall(route, [c for c in EXTREME if c[3] <= 64]) == [3, 3, 3]


def test_prefill_kernels_of_the_matmul_tests(route):
    """test_gpu_matmul.py's tests of the 8-wave and the decoded slabs, and its
    512-token layer (gate alone too)."""
    q4, q5, q6 = TYPE_Q4_K, TYPE_Q5_K, TYPE_Q6_K
    assert _prefill(route, [(q4, [9728, 9728], 2560, 512), (q4, [13200, 13107], 512, 300)]) == ["B", "B"]
    assert _prefill(route, [(q5, [2048, 512, 528], 2560, 256), (q5, [4000, 1037], 1024, 333), (q6, [3000, 450], 1024, 384),
                            (q6, [2560], 4352, 129), (q5, [9000], 2560, 65), (q5, [9000], 2560, 100)]) == ["D"] * 6
    assert _prefill(route, [(q5, [6144], 2560, 512), (q4, [2560], 4096, 512), (q6, [2560], 9728, 512)]) == ["C", "P", "E"]


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


def _tall(route, cases):
    return [int(v) for v in route([f"tall {FORMAT[t]} {rows} {K} {M} 256" for t, rows, K, M in cases])]


def test_tall_kernels_of_the_gpu_cases(route):
    cases = [(t, sum(64 * -(-n // 64) for n in rows), K, M) for t, rows, K, M, _ in TALL]
    assert _tall(route, cases) == [(c[3] + 15) // 16 for c in cases]


def test_tall_wave_slabs_only_where_faster(route):
    """Not under one workgroup of 64 rows per CU, not where the last round is too
    empty for the K, and at 32 tokens or fewer not at the K that the part kernel
    reads best (all of these measured slower than the small-M kernels)."""
    q4, q5, q6 = TYPE_Q4_K, TYPE_Q5_K, TYPE_Q6_K
    slower = [(q4, 9728, 2560, 64), (q4, 18432, 2560, 49), (q5, 18432, 2560, 33), (q5, 19456, 2560, 33),
              (q6, 18432, 2560, 64), (q6, 19456, 3072, 64), (q4, 16384, 3072, 33), (q4, 33000, 9728, 33), (q4, 19456, 9728, 49),
              (q4, 33000, 2560, 17), (q4, 38000, 3072, 32), (q4, 49300, 3072, 24), (q6, 66000, 3072, 12),
              (q6, 151936, 2560, 16), (q6, 100000, 2048, 9)]
    assert _tall(route, slower) == [0] * len(slower)
    faster = [(q4, 28672, 2560, 64), (q4, 19456, 2560, 37), (q6, 19456, 2560, 48), (q5, 16384, 2560, 49),
              (q6, 18432, 4096, 49), (q5, 17408, 8192, 33),
              (q4, 33000, 4096, 17), (q4, 44000, 2560, 24), (q6, 151936, 1024, 16), (q6, 100000, 4096, 9),
              (q6, 18432, 1024, 33)]
    assert _tall(route, faster) == [(c[3] + 15) // 16 for c in faster]
