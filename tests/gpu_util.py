"""Helpers for the GPU parity tests."""
import numpy as np

# stated tolerance for fp32 dot / GEMM outputs: max|y - ref| / max|ref|
TOL = 1e-3


def norm_err(y, ref) -> float:
    y = np.asarray(y, np.float64)
    ref = np.asarray(ref, np.float64)
    scale = np.abs(ref).max()
    return float(np.abs(y - ref).max() / (scale if scale > 0 else 1.0))


def check_outputs(y, ref, what=""):
    """Within the stated tolerance, and — by construction of the kernels —
    equal to the reference's fp32 sums bit for bit."""
    y = np.ascontiguousarray(y, np.float32)
    ref = np.ascontiguousarray(ref, np.float32)
    assert y.shape == ref.shape, (what, y.shape, ref.shape)
    err = norm_err(y, ref)
    assert err <= TOL, f"{what}: normalized max error {err:.3e} > {TOL}"
    nbad = int(np.count_nonzero(y.view(np.uint32) != ref.view(np.uint32)))
    assert nbad == 0, f"{what}: {nbad} of {y.size} outputs differ in bits (norm err {err:.3e})"


def check_q8k(ctx, oracle, buf, M, K, y):
    """Every section of a device Q8_K buffer against the oracle's quantizer on
    the fp32 rows y [M][K], bit for bit."""
    d, qs, bs = ctx.read_q8k(buf, M, K)
    ed, eqs, ebs = oracle.quantize_q8k(y)
    assert np.array_equal(d.view(np.uint32), ed.view(np.uint32)), "scales"
    assert np.array_equal(qs, eqs) and np.array_equal(bs, ebs), "codes and sums of 32"
    assert np.array_equal(ctx.read_q8k_tiles(buf, M, K), eqs), "tiles section"
    assert np.array_equal(ctx.read_q8k_h(buf, M, K), oracle.f32_to_fp16(y)), "h section"
    assert np.array_equal(ctx.read_q8k_bh(buf, M, K),
                          eqs.reshape(M, K // 16, 16).astype(np.int32).sum(axis=2).astype(np.float32)), "sums of 16"


def say(msg):
    print(f"[gpu-case] {msg}", flush=True)
