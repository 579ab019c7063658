"""GPU parity of gemm_few_kernel (few rows, K interleaved over the waves of a workgroup) against the CPU oracle.

Both column widths, one and two row groups, the row counts at their edges, both weight formats and every
epilogue; K that gives some waves no step, a last partial ring of steps and several rings; columns that are
no multiple of the width.  Exact.
"""
import numpy as np
import pytest

from rknpu2_matmul_open_amd import capi, ops, workloads

pytestmark = pytest.mark.gpu

# (rows, columns, K): int8 weights; 16 columns up to 4096, 32 beyond
INT8 = [(9, 100, 40), (16, 4096, 300), (13, 513, 2100), (17, 1999, 2050), (32, 4095, 700), (9, 4200, 300), (16, 4129, 2500),
        (17, 5000, 600), (32, 4128, 1111), (33, 4200, 300), (64, 4133, 1300), (56, 8300, 520),
        (5, 300, 8192), (8, 100, 9000), (3, 70, 17000), (2, 4200, 17000)]
INT4 = [(9, 100, 40), (16, 4096, 300), (13, 513, 2100), (17, 1999, 2050), (32, 4032, 700), (5, 300, 4200), (8, 128, 9000),
        (3, 70, 9000), (2, 64, 17000)]


@pytest.mark.parametrize("M,N,K", INT8)
@pytest.mark.parametrize("kind", ["f16", "f32", "i32"])
def test_int8_weights(sess, oracle, M, N, K, kind):
    c = workloads.w8a8_case(M, K, N, seed_w=M + N, seed_a=K)
    if kind == "i32":
        A = np.random.default_rng(M).integers(-128, 128, (M, K)).astype(np.int8)
        op, dtype = ops.W8A8Linear(sess, capi.I8I8I32, M, c["B"]), np.int32
        want = oracle.gemm_i8(A, c["B"])
    elif kind == "f16":
        A = c["A"]
        op, dtype = ops.W8A8Linear(sess, capi.F16I8F16_DYNAMIC, M, c["B"], c["w_scale"]), np.uint16
        want = oracle.w8a8(A, c["B"], c["w_scale"])["C"]
    else:
        A = workloads.normal_f32(K, (M, K))
        op, dtype = ops.W8A8Linear(sess, capi.F32I8F32_DYNAMIC, M, c["B"], c["w_scale"]), np.float32
        want = oracle.w8a8(A, c["B"], c["w_scale"])["C"]
    dA, dC = sess.to_device(A), sess.empty_device(M * N * np.dtype(dtype).itemsize)
    try:
        for _ in range(2):
            assert op.run_device(dA, dC) == 0
            assert sess.sync() == 0
            got = sess.from_device(dC, (M, N), dtype)
            assert np.array_equal(got.view(np.uint8), np.ascontiguousarray(want, dtype).view(np.uint8))
    finally:
        sess.free_device(dA)
        sess.free_device(dC)
        op.close()


@pytest.mark.parametrize("M,N,K", INT4)
@pytest.mark.parametrize("kind", ["f16", "f32", "i32"])
def test_int4_weights(sess, oracle, M, N, K, kind):
    c = workloads.w4a8_case(M, K, N, seed_w=N, seed_a=M)
    w = ops.W4A8Weights(sess, c["B"], c["w_scale"])
    ws = ops.W4A8Workspace(sess, M, N, K)
    A = oracle.half_to_float(c["A"]).astype(np.float32).reshape(M, K)
    try:
        if kind == "f16":
            rc, got = ws.run_f16(w, c["A"])
            want = oracle.w4a8(c["A"], c["B"], c["w_scale"])["C"]
        elif kind == "f32":
            rc, got = ws.run_f32(w, A)
            want = oracle.w4a8(A, c["B"], c["w_scale"])["C"]
        else:
            rc, got = ws.run_i32(w, A)
            want = oracle.w4a8(A, c["B"], c["w_scale"])["acc"]
        assert rc == 0
        assert np.array_equal(got.view(np.uint8), np.ascontiguousarray(want, got.dtype).view(np.uint8))
    finally:
        ws.close()
        w.close()
