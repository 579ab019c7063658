"""GPU parity of the row quantization where its workgroups are dealt to the dies, against the CPU oracle.

Workgroups take rows (or four rows, or parts of a row) in one contiguous range per die: row counts below, at
and around multiples of eight and of 8 x 4, rows of less than a chunk and with a ragged last chunk, the line
between one row and four rows per workgroup (at 513 for fp32 rows that are not 16-byte aligned), and, for the
re-quantized middle of an FFN, the wave-per-row kernel (up to 4096 columns) and rows shared by two to eight
workgroups.  Exact.
"""
import numpy as np
import pytest

from rknpu2_matmul_open_amd import capi, ops, workloads

pytestmark = pytest.mark.gpu

SHAPES = [(9, 40), (15, 2050), (33, 16400), (67, 300), (255, 2049), (256, 2030), (257, 2048), (767, 2033), (768, 2048),
          (512, 2051), (513, 2051)]


@pytest.mark.parametrize("M,K", SHAPES)
@pytest.mark.parametrize("kind", ["f16", "f32", "i32"])
def test_rows(sess, oracle, M, K, kind):
    N = 64
    c = workloads.w8a8_case(M, K, N, seed_w=M, seed_a=K)
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
        assert op.run_device(dA, dC) == 0
        assert sess.sync() == 0
        got = sess.from_device(dC, (M, N), dtype)
        assert np.array_equal(got.view(np.uint8), np.ascontiguousarray(want, dtype).view(np.uint8))
    finally:
        sess.free_device(dA)
        sess.free_device(dC)
        op.close()


@pytest.mark.parametrize("M,I", [(9, 992), (64, 992), (65, 1024), (131, 4096), (33, 4128), (70, 8224), (513, 4160)])
def test_middle_of_an_ffn(sess, oracle, M, I):
    H = 96
    gu = workloads.w4a8_case(M, H, 2 * I, seed_w=I, seed_a=M)
    dn = workloads.w4a8_case(M, I, H, seed_w=I + 1, seed_a=M)
    A = workloads.normal_f32(M, (M, H))
    gu_w, dn_w = ops.W4A8Weights(sess, gu["B"], gu["w_scale"]), ops.W4A8Weights(sess, dn["B"], dn["w_scale"])
    gu_ws, dn_ws = ops.W4A8Workspace(sess, M, 2 * I, H), ops.W4A8Workspace(sess, M, H, I)
    try:
        rc, middle, out = ops.w4a8_ffn(sess, gu_ws, gu_w, dn_ws, dn_w, A)
        want = oracle.w4a8_ffn(A, gu["B"], gu["w_scale"], dn["B"], dn["w_scale"])
        assert rc == 0
        assert np.array_equal(middle.view(np.uint32), np.asarray(want["middle"], np.float32).view(np.uint32))
        assert np.array_equal(out.view(np.uint32), np.asarray(want["C"], np.float32).view(np.uint32))
    finally:
        for h in (gu_ws, dn_ws, gu_w, dn_w):
            h.close()


@pytest.mark.parametrize("M,K", [(9, 16384), (9, 4097), (33, 4111), (64, 8193), (65, 8193), (64, 12289), (128, 4112), (129, 4112),
                                 (128, 8208), (40, 16385)])
def test_long_rows_shared_by_workgroups(sess, oracle, M, K):
    """Scanned rows of more than 256 chunks: two or four workgroups each (the last part whole, one chunk, or without
    any), the row counts where that ends, rows too long for it; a value that is not finite in the last part."""
    N = 64
    c = workloads.w4a8_case(M, K, N, seed_w=M, seed_a=K)
    w, ws = ops.W4A8Weights(sess, c["B"], c["w_scale"]), ops.W4A8Workspace(sess, M, N, K)
    A = c["A"].copy()
    try:
        for dtype in (np.uint16, np.float32):
            X = A if dtype is np.uint16 else oracle.half_to_float(A).astype(np.float32).reshape(M, K)
            # (the largest value of a row in one part, of the next row in another)
            X[np.arange(M), (np.arange(M) * 4099 + K - 1) % K] = 0x5500 if dtype is np.uint16 else 80.0
            dA, dC = sess.to_device(X), sess.empty_device(M * N * X.itemsize)
            run = sess.lib.rk_npu_w4a8_run_f16_device if dtype is np.uint16 else sess.lib.rk_npu_w4a8_run_f32_device
            assert run(ws.h, w.h, dA, dC) == 0 and sess.sync() == 0
            got = sess.from_device(dC, (M, N), dtype)
            want = oracle.w4a8(X, c["B"], c["w_scale"])["C"]
            assert np.array_equal(got.view(np.uint8), np.ascontiguousarray(want, dtype).view(np.uint8))
            sess.free_device(dA)
            X = X.copy()
            X[M - 1, K - 1] = 0x7c00 if dtype is np.uint16 else np.inf
            dA = sess.to_device(X)
            assert run(ws.h, w.h, dA, dC) == 0 and sess.sync() == capi.RK_NPU_ERR_PARAM
            sess.free_device(dA)
            sess.free_device(dC)
    finally:
        ws.close()
        w.close()
