"""The wave-slab GEMM (csrc/qmm_wslab.hip) vs the oracle, bit for bit: its
prefill shapes (128 rows x 96 tokens, 128 x 64, 64 x 64) and its tall ones (up
to 64 tokens) on every k-quant format, with rows and tokens past the last tile,
one block and several, a task group, a residual, extreme scales, and Q6_K rows
off every 16-B boundary."""
import numpy as np
import pytest

import qmm_hip
import synth
from gpu_util import check_outputs, say
from oracle import TYPE_Q4_K, TYPE_Q5_K, TYPE_Q6_K
from test_gpu_matmul import _extreme_weights as extreme_weights

pytestmark = pytest.mark.gpu


def _run(ctx, oracle, type_id, rows, K, M, residual, skip=0):
    say(f"type {type_id} rows={rows} K={K} M={M} residual={residual} from row {skip}")
    x = synth.activations(M, K, seed=K + M)
    xb = ctx.upload(x)
    rb = qmm_hip.row_bytes(type_id, K)
    bufs, tasks, ref = [xb], [], []
    for i, N in enumerate(rows):
        w = synth.weights(type_id, N + skip, K, seed=31 * i + N)
        wb, yb = ctx.weight_upload(w, type_id, N + skip, K), ctx.malloc(M * N * 4)
        res = synth.activations(M, N, seed=7 * i + N) if residual else None
        resb = ctx.upload(res) if residual else None
        bufs += [b for b in (wb, yb, resb) if b is not None]
        tasks.append(qmm_hip.MatrixTask(wb.ptr + skip * rb, type_id, N, K, yb, N, resb, N if residual else 0))
        ref.append(dict(w=w[skip * rb:], type=type_id, rows=N, **(dict(residual=res) if residual else {})))
    ctx.gemm_multi_dispatch(xb, M, K, tasks)
    ctx.sync()
    for t, r in zip(tasks, oracle.gemm_multi(x, ref)):
        check_outputs(ctx.d2h(t.dst, np.float32, (M, t.rows)), r, f"rows={t.rows} K={K} M={M}")
    for b in bufs:
        ctx.free(b)


# kernel (csrc/qmm_route.h): cases that take it at 256 CUs (tests/test_route.py checks that they do)
PREFILL = {
    # 128 rows x 96 tokens: ragged last tokens (80, 40, 70 of 96) and rows
    "A": [(TYPE_Q4_K, [3000], 512, 2000, True), (TYPE_Q6_K, [5001], 768, 1000, False), (TYPE_Q5_K, [4100], 256, 1030, True),
          (TYPE_Q5_K, [6100], 256, 2000, False)],
    # 128 x 64
    "B": [(TYPE_Q4_K, [5003], 768, 700, False), (TYPE_Q6_K, [6001], 512, 600, True), (TYPE_Q5_K, [6100], 256, 600, False),
          (TYPE_Q5_K, [6020, 75], 512, 590, True)],
    # 64 x 64: one token past a group, a 49-row task in the group
    "C": [(TYPE_Q4_K, [8190], 256, 257, True), (TYPE_Q5_K, [8201], 512, 300, False), (TYPE_Q6_K, [9001], 768, 300, False),
          (TYPE_Q4_K, [2500, 49], 512, 1000, True)],
    # Q6_K decoded slabs of 32 rows x 256 tokens: odd and even step counts, ragged rows and tokens
    "E": [(TYPE_Q6_K, [4096], 4352, 512, False), (TYPE_Q6_K, [2003], 4608, 1000, True),
          (TYPE_Q6_K, [6100, 900], 4352, 250, False), (TYPE_Q6_K, [4090], 512, 509, True)],
}


@pytest.mark.parametrize("type_id,rows,K,M,residual", PREFILL["A"] + PREFILL["B"] + PREFILL["C"])
def test_wave_slabs(ctx, oracle, type_id, rows, K, M, residual):
    _run(ctx, oracle, type_id, rows, K, M, residual)


@pytest.mark.parametrize("type_id,rows,K,M,residual", PREFILL["E"])
def test_decoded_slabs_256_tokens(ctx, oracle, type_id, rows, K, M, residual):
    """Q6_K decoded slabs of 32 rows x 256 tokens (csrc/qmm_slab.hip)."""
    _run(ctx, oracle, type_id, rows, K, M, residual)


# 64 rows x 64, 48, 32 and 16 tokens: one block (fewer than the stages), two, three and more; ragged tokens and rows
TALL = [
    (TYPE_Q4_K, [16400], 256, 64, True), (TYPE_Q5_K, [20001], 512, 50, False), (TYPE_Q6_K, [19000], 768, 49, False),
    (TYPE_Q4_K, [9728, 9700], 1280, 37, True), (TYPE_Q5_K, [19456], 256, 48, False), (TYPE_Q6_K, [20003], 512, 33, True),
    (TYPE_Q4_K, [30000], 768, 17, False), (TYPE_Q4_K, [29001], 256, 32, True),
    (TYPE_Q6_K, [65600], 256, 9, True), (TYPE_Q6_K, [65537], 768, 16, False)]


@pytest.mark.parametrize("type_id,rows,K,M,residual", TALL)
def test_wave_slabs_tall(ctx, oracle, type_id, rows, K, M, residual):
    _run(ctx, oracle, type_id, rows, K, M, residual)


# taller than the small-M and the other prefill kernels: tall slabs, and 128 x 96 / 64 x 64
EXTREME = [(TYPE_Q4_K, 16400, 512, 40), (TYPE_Q5_K, 16400, 512, 40), (TYPE_Q6_K, 16400, 512, 40),
           (TYPE_Q4_K, 3000, 512, 2000), (TYPE_Q5_K, 8201, 512, 300), (TYPE_Q6_K, 9001, 768, 300)]


@pytest.mark.parametrize("type_id,rows,K,M", EXTREME)
def test_wave_slabs_extreme_scales(ctx, oracle, type_id, rows, K, M):
    """The largest scales, mins and quants: the integer sums stay exact."""
    say(f"extreme scales type {type_id} rows={rows} K={K} M={M}")
    w = extreme_weights(type_id, rows, K, seed=rows + M)
    x = synth.activations(M, K, seed=701)
    x[:, ::7] *= 50.0   # large entries: many codes at +-127
    wb = ctx.weight_upload(w, type_id, rows, K)
    y = ctx.gemm(type_id, wb, rows, K, x)
    ctx.free(wb)
    check_outputs(y, oracle.gemm_multi(x, [dict(w=w, type=type_id, rows=rows)])[0], f"extreme {type_id} M={M}")


@pytest.mark.parametrize("rows,K,M", [([20000], 768, 40), ([66000], 768, 12), ([5000], 768, 1000), ([6000], 256, 600), ([9000], 768, 300)])
def test_wave_slabs_unaligned_q6k(ctx, oracle, rows, K, M):
    """Q6_K rows from row 1 of a tensor: 210-B blocks 2 B off a 4-B boundary."""
    _run(ctx, oracle, TYPE_Q6_K, rows, K, M, False, skip=1)
