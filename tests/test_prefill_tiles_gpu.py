"""The prefill matmuls' tiles (gemm.hip, gemm_cq.hip): each tile a launch can
choose, at ragged token counts, rows and group counts, bit-identical with the
oracle's MatMulRows; exponent-31 norms, row ranges, batches whose jobs end
inside a tile, and activations that are not 16-byte aligned."""
import numpy as np
import pytest

from test_gemm_gpu import run_fused
from test_matmul_batch_gpu import run_batch
from test_matmul_gpu import SENTINEL, cq_case, hip_book, int8_case, run_i8

pytestmark = pytest.mark.gpu


def run_cq(hip, case, rows, cols, bits, tokens, ldy, r0, r1, shift=0):
    weights = hip.Weights.codebook(case["indices"], case["norms"], hip_book(hip, case["book"]), rows, cols, bits)
    v = np.zeros(tokens * cols + shift, dtype=np.int8)
    v[shift:] = np.asarray(case["values"], dtype=np.int8).reshape(-1)[:tokens * cols]
    dq = hip.DeviceBuffer.from_array(v)
    ds, do = hip.DeviceBuffer.from_array(case["scales"]), hip.DeviceBuffer.from_array(case["offsets"])
    dy = hip.DeviceBuffer.from_array(np.full(tokens * ldy, SENTINEL, dtype=np.float32))
    hip.check(hip.lib().nhip_matmul_cq_dev(weights.handle, dq.ptr + shift, ds.ptr, do.ptr, case["act"].stride, tokens,
                                           dy.ptr, ldy, r0, r1, None))
    return dy.download(np.float32)


def oracle_cq(orc, case, tokens, ldy, r0, r1):
    want = np.full(tokens * ldy, SENTINEL, dtype=np.float32)
    orc.matmul_rows(case["cq"], case["act"], tokens, want, ldy, r0, r1)
    return want


@pytest.mark.parametrize("bits", [2, 4])
@pytest.mark.parametrize("tokens,rows,cols", [
    (17, 16, 128),      # 16 x 64: one tile, one group
    (31, 70, 384),      # an odd group count, a last workgroup of one tile
    (64, 130, 256),
    (250, 3067, 128),   # 32 x 64
    (97, 8200, 384),
    (500, 3063, 256),   # 64 x 128
    (449, 3100, 640),
])
def test_codebook_tiles_bit_exact(hip, orc, bits, tokens, rows, cols):
    case = cq_case(orc, tokens + rows + bits, rows, cols, bits, tokens)
    got = run_cq(hip, case, rows, cols, bits, tokens, rows, 0, rows)
    assert np.array_equal(got.view(np.uint32), oracle_cq(orc, case, tokens, rows, 0, rows).view(np.uint32))


@pytest.mark.parametrize("bits", [2, 4])
@pytest.mark.parametrize("r0,r1,shift", [(5, 77, 0), (79, 80, 0), (16, 32, 8), (0, 80, 8)])
def test_codebook_row_ranges_and_alignment(hip, orc, bits, r0, r1, shift):
    tokens, rows, cols = 40, 80, 256
    case = cq_case(orc, 40 + r0 + bits, rows, cols, bits, tokens)
    got = run_cq(hip, case, rows, cols, bits, tokens, rows + 3, r0, r1, shift)
    assert np.array_equal(got.view(np.uint32), oracle_cq(orc, case, tokens, rows + 3, r0, r1).view(np.uint32))


@pytest.mark.parametrize("bits", [2, 4])
@pytest.mark.parametrize("tokens,rows", [(60, (37, 100, 5, 40)), (500, (2999, 37, 100, 40))])
def test_codebook_batch_jobs_end_inside_a_tile(hip, orc, bits, tokens, rows):
    cols = 384
    cases = [cq_case(orc, 70 + j + bits, r, cols, bits, tokens) for j, r in enumerate(rows)]
    a = cases[0]
    cases[2]["norms"].reshape(-1)[::3] = 0x7C01  # exponent 31 in one job (the oracle reads the same array)
    weights = [hip.Weights.codebook(c["indices"], c["norms"], hip_book(hip, c["book"]), r, cols, bits)
               for c, r in zip(cases, rows)]
    got = run_batch(hip, [w.handle for w in weights], rows, a["values"], a["scales"], a["offsets"], a["act"].stride,
                    tokens)
    for j, (c, r) in enumerate(zip(cases, rows)):
        want = np.full(tokens * (r + 3), SENTINEL, dtype=np.float32)
        orc.matmul_rows(c["cq"], a["act"], tokens, want, r + 3, 0, r)
        assert np.array_equal(got[j].reshape(-1).view(np.uint32), want.view(np.uint32)), j


@pytest.mark.parametrize("tokens,rows,cols", [
    (17, 16, 32),       # 16 x 64: one tile, one group
    (20, 70, 288),      # a partial last stage
    (250, 4099, 96),    # 32 x 64
    (1000, 4090, 288),  # 64 x 128
    # row blocks not a multiple of 8, renumbered over the XCDs: each tile
    (33, 2300, 4096), (250, 4099, 608), (1000, 4500, 480),
])
def test_int8_tiles_bit_exact(hip, orc, tokens, rows, cols):
    w, scales, x, q, qs = int8_case(orc, tokens + rows, rows, cols, tokens)
    weights = hip.Weights.int8(w, scales)
    want = np.full((tokens, rows), SENTINEL, dtype=np.float32)
    orc.matmul_rows_i8(w, scales, q, qs, tokens, want, rows, 0, rows)
    y = run_i8(hip, weights, q, qs, tokens, rows, 0, rows)
    assert np.array_equal(y.view(np.uint32), want.view(np.uint32))
    # the fused epilogue rounds once per group instead of twice: the entry's
    # stated bound
    yf = run_fused(hip, weights, q, qs, tokens, rows, 0, rows)
    assert np.max(np.abs(yf.astype(np.float64) - want)) <= 1e-4 * float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))


@pytest.mark.parametrize("shift", [4, 8])
@pytest.mark.parametrize("tokens,rows,cols", [(3, 64, 1024), (17, 70, 96), (31, 100, 288), (64, 130, 256), (200, 48, 2048)])
def test_int8_activations_off_16_bytes(hip, orc, tokens, rows, cols, shift):
    """Activations 4 or 8 bytes past a 16-byte boundary: both entries run in
    the reference's order, in the kernels that load them through registers."""
    w, scales, x, q, qs = int8_case(orc, tokens + rows + shift, rows, cols, tokens)
    weights = hip.Weights.int8(w, scales)
    want = np.full((tokens, rows), SENTINEL, dtype=np.float32)
    orc.matmul_rows_i8(w, scales, q, qs, tokens, want, rows, 0, rows)
    v = np.zeros(tokens * cols + shift, dtype=np.int8)
    v[shift:] = q.reshape(-1)
    dq, ds = hip.DeviceBuffer.from_array(v), hip.DeviceBuffer.from_array(qs)
    lib = hip.lib()
    for entry in (lib.nhip_matmul_i8_dev, lib.nhip_matmul_i8_fused_dev):
        dy = hip.DeviceBuffer.from_array(np.full(tokens * rows, SENTINEL, dtype=np.float32))
        hip.check(entry(weights.handle, dq.ptr + shift, ds.ptr, tokens, dy.ptr, rows, 0, rows, None))
        assert np.array_equal(dy.download(np.float32).view(np.uint32), want.reshape(-1).view(np.uint32))
