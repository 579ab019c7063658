"""GPU parity of the LDS-ring GEMM's K loop against the CPU oracle: every tile shape of gemm_wk_kernel with K from less than
one block of 256 to more than a trip of the unrolled loop, so that each remainder of the trip (0 .. 7 steps) and K that ends
inside a step occurs; rows and columns end inside a tile.  (gemm_wk_big_kernel: tests/test_gpu_large_tiles.py.)  Integer
sums and a fixed order of the floating-point steps: exact.
"""
import ctypes as C

import numpy as np
import pytest

from rknpu2_matmul_open_amd import capi, ops, workloads

pytestmark = pytest.mark.gpu

NARROW, TILES = 4, 5  # rkh_gemm_kernel
KS = (130, 256, 500, 768, 1024, 1200, 1500, 1792, 2048, 2300)
I32, F16, SWIGLU = 0, 1, 3


def _route(M, N, K, w4, epi):
    v = [C.c_int() for _ in range(5)]
    assert capi.load_library().rkh_gemm_route(M, N, K, w4, epi, *[C.byref(x) for x in v]) == 0
    return v[0].value, v[1].value


@pytest.mark.parametrize("K", KS)
@pytest.mark.parametrize("M,N,kernel,rows", [(129, 4100, NARROW, 64), (1000, 2500, NARROW, 128), (1800, 2900, TILES, 128)])
def test_int8_weights(sess, oracle, M, N, K, kernel, rows):
    assert _route(M, N, K, 0, I32) == (kernel, rows)
    rng = np.random.default_rng(K)
    A, B = rng.integers(-128, 128, (M, K)).astype(np.int8), rng.integers(-128, 128, (K, N)).astype(np.int8)
    op = ops.W8A8Linear(sess, capi.I8I8I32, M, B)
    try:
        rc, got = op.run(A)
        assert rc == 0 and np.array_equal(got, oracle.gemm_i8(A, B))
    finally:
        op.close()


@pytest.mark.parametrize("K", KS)
@pytest.mark.parametrize("M,N,epi,kernel,rows", [(129, 4100, F16, NARROW, 64), (700, 3000, F16, TILES, 64), (1800, 2304, F16, TILES, 128),
                                                 (300, 6016, SWIGLU, TILES, 32), (900, 4032, SWIGLU, TILES, 64)])
def test_int4_weights(sess, oracle, one_piece, M, N, K, epi, kernel, rows):
    assert _route(M, N, K, 1, epi) == (kernel, rows)
    c = workloads.w4a8_case(M, K, N, seed_w=K, seed_a=M)
    w = ops.W4A8Weights(sess, c["B"], c["w_scale"])
    ws = ops.W4A8Workspace(sess, M, N, K)
    try:
        if epi == F16:
            (rc, got), _ = one_piece(lambda: ws.run_f16(w, c["A"]))
            want = oracle.w4a8(c["A"], c["B"], c["w_scale"])["C"]
        else:
            A32 = oracle.half_to_float(c["A"]).astype(np.float32).reshape(M, K)
            (rc, got), _ = one_piece(lambda: ws.run_swiglu_f32(w, A32))
            want = oracle.w4a8_swiglu(A32, c["B"], c["w_scale"])["middle"]
        assert rc == 0 and np.array_equal(got.view(np.uint8), np.ascontiguousarray(want, got.dtype).view(np.uint8))
    finally:
        ws.close()
        w.close()


# Exact products of 64- and 128-row tiles read the caller's int8 rows where these allow 16-byte pieces: K that ends in a step's
# first piece, at its end and, with steps of 128 k, one whole step before the padded end; a last row block of one row
@pytest.mark.parametrize("K", [16, 128, 144, 256, 272, 1040, 1536, 40])
@pytest.mark.parametrize("M,N,rows,offset", [(129, 4100, 64, 0), (129, 4100, 64, 16), (129, 4100, 64, 4), (1000, 2500, 128, 0), (897, 2500, 128, 32)])
def test_rows_as_given(sess, oracle, M, N, K, rows, offset):
    assert _route(M, N, K, 0, I32) == (NARROW, rows)
    rng = np.random.default_rng(K + M)
    A, B = rng.integers(-128, 128, (M, K)).astype(np.int8), rng.integers(-128, 128, (K, N)).astype(np.int8)
    op = ops.W8A8Linear(sess, capi.I8I8I32, M, B)
    base = sess.to_device(np.concatenate([np.zeros(offset, np.int8), A.reshape(-1)]))
    dC = sess.empty_device(M * N * 4)
    try:
        kernels = [name for name, _ in ops.profile_kernels(sess, lambda: op.run_device(base + offset, dC), 1, 1)]
        assert ("quant_rows_kernel" in kernels) == (K % 16 != 0 or offset % 16 != 0), kernels
        want = oracle.gemm_i8(A, B)
        assert np.array_equal(sess.from_device(dC, (M, N), np.int32), want)
        q, s = np.empty((M, K), np.int8), np.empty(M, np.float32)
        assert sess.lib.rk_npu_matmul_workspace_read_quantized(op.ws, capi.ptr(q), capi.ptr(s)) == 0
        assert np.array_equal(q, A)
        assert sess.lib.rk_npu_matmul_workspace_rerun_gemm_device(op.ws, op.w, dC) == 0 and sess.sync() == 0
        assert np.array_equal(sess.from_device(dC, (M, N), np.int32), want)
    finally:
        sess.free_device(base)
        sess.free_device(dC)
        op.close()


# The tiles that such a call owes its workspace, 9 .. 32 to a workgroup: two, three and four to a wave, up to the most that a
# wave takes; beyond it the rows are re-tiled by a launch of their own
@pytest.mark.parametrize("M,N,K,rows,share", [(600, 500, 752, 64, 12), (600, 500, 1040, 64, 20), (600, 500, 1792, 64, 28), (600, 500, 2048, 64, 32),
                                              (600, 384, 1536, 64, 32), (600, 500, 2064, 64, 36), (300, 4096, 14336, 64, 28),
                                              (2500, 1000, 752, 128, 12), (2500, 1000, 1264, 128, 20), (2500, 1000, 1792, 128, 28),
                                              (2500, 1000, 2048, 128, 32), (2500, 1000, 2064, 128, 36)])
def test_tiles_owed_to_the_workspace(sess, oracle, M, N, K, rows, share):
    assert _route(M, N, K, 0, I32) == (NARROW, rows)
    assert -(-(rows // 32 * ((K + 255) // 256 * 8)) // -(-N // 128)) == share
    rng = np.random.default_rng(K)
    B = rng.integers(-128, 128, (K, N)).astype(np.int8)
    op = ops.W8A8Linear(sess, capi.I8I8I32, M, B)
    dA, dC = sess.empty_device(M * K), sess.empty_device(M * N * 4)
    try:
        for _ in range(2):  # (the second call's rows take the place of the first one's)
            A = rng.integers(-128, 128, (M, K)).astype(np.int8)
            assert sess.lib.rk_npu_hip_upload(sess.ctx, dA, capi.ptr(A), A.nbytes) == 0
            kernels = [name for name, _ in ops.profile_kernels(sess, lambda: op.run_device(dA, dC), iters=1, warmup=0)]
            assert ("quant_rows_kernel" in kernels) == (share > 32), kernels
            want = oracle.gemm_i8(A, B)
            assert np.array_equal(sess.from_device(dC, (M, N), np.int32), want)
            q = np.empty((M, K), np.int8)
            assert sess.lib.rk_npu_matmul_workspace_read_quantized(op.ws, capi.ptr(q), None) == 0
            assert np.array_equal(q, A)
        assert sess.lib.rk_npu_matmul_workspace_rerun_gemm_device(op.ws, op.w, dC) == 0 and sess.sync() == 0
        assert np.array_equal(sess.from_device(dC, (M, N), np.int32), want)
    finally:
        sess.free_device(dA)
        sess.free_device(dC)
        op.close()


def test_a_result_over_the_rows(sess, oracle):
    """The result may be written over the rows it is made of: they are copied first then, down to 16 common bytes on
    either side, and are not where one ends as the other begins.  (The values alone would not show it: the few
    workgroups of this size read all their rows before any of them writes.)"""
    M, N, K = 129, 4100, 512
    rng = np.random.default_rng(7)
    A, B = rng.integers(-128, 128, (M, K)).astype(np.int8), rng.integers(-128, 128, (K, N)).astype(np.int8)
    op = ops.W8A8Linear(sess, capi.I8I8I32, M, B)
    want = oracle.gemm_i8(A, B)
    a, c = A.nbytes, M * N * 4
    buf = sess.empty_device(a + c)
    try:
        for rows_at, result_at, apart in ((0, 0, False), (1024, 0, False), (0, a - 16, False), (c - 16, 0, False), (0, a, True), (c, 0, True)):
            assert sess.lib.rk_npu_hip_upload(sess.ctx, buf + rows_at, capi.ptr(A), a) == 0
            kernels = [name for name, _ in ops.profile_kernels(sess, lambda: op.run_device(buf + rows_at, buf + result_at), iters=1, warmup=0)]
            assert ("quant_rows_kernel" in kernels) == (not apart), (rows_at, result_at, kernels)
            assert np.array_equal(sess.from_device(buf + result_at, (M, N), np.int32), want)
    finally:
        sess.free_device(buf)
        op.close()


# K split over workgroups: the reduce launch takes the 64 rows that a wave of a 128-row tile kept in two halves; rows that end in
# either half of either wave, at its edges, and with the tile
@pytest.mark.parametrize("M", [673, 704, 705, 737, 767, 768])
@pytest.mark.parametrize("kind", [capi.I8I8I32, capi.F16I8F16_DYNAMIC, capi.F32I8F32_DYNAMIC])
def test_k_split_of_128_row_tiles(sess, oracle, one_piece, M, kind):
    N, K = 700, 10240
    assert _route(M, N, K, 0, I32 if kind == capi.I8I8I32 else F16) == (TILES, 128)
    c = workloads.w8a8_case(M, K, N, seed_w=N, seed_a=M)
    if kind == capi.I8I8I32:
        A, scale = np.random.default_rng(M).integers(-128, 128, (M, K)).astype(np.int8), None
        want = oracle.gemm_i8(A, c["B"])
    else:
        A, scale = (c["A"] if kind == capi.F16I8F16_DYNAMIC else workloads.normal_f32(M, (M, K))), c["w_scale"]
        want = oracle.w8a8(A, c["B"], scale)["C"]
    op = ops.W8A8Linear(sess, kind, M, c["B"], scale)
    try:
        (rc, got), kernels = one_piece(lambda: op.run(A))
        assert rc == 0 and kernels[-1] == "gemm_wk_reduce_kernel"
        assert np.array_equal(got.view(np.uint8), np.ascontiguousarray(want, got.dtype).view(np.uint8))
    finally:
        op.close()
