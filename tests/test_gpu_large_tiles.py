"""GPU parity of the 256 x 256 tiles of the large-tile GEMM (gemm_wk_big_kernel) against the CPU oracle.

The kernel serves dense calls with more than 256 tiles of 128 x 256; the cases put the places where it can
go wrong into small problems: rows that end in a strip of 128-row tiles, in a partly filled 256-row tile or
exactly, a last round cut into halves with and without a strip behind them (tests/test_plan_cpu.py holds the cut
of each shape), one and several trips of the unrolled K loop with and without a
remainder, columns that are no multiple of anything, and every epilogue.  Integer sums and a fixed order of
the floating-point steps: exact.
"""
import ctypes as C

import numpy as np
import pytest

from rknpu2_matmul_open_amd import capi, ops, workloads

pytestmark = pytest.mark.gpu

SHAPES = [(1100, 7500, 200),    # strip of 76 rows; one partial trip of the K loop
          (1224, 7457, 300),    # last 256-row tile with 200 rows; odd columns
          (2816, 6656, 513),    # 286 tiles of 256 x 256, two rounds of them; K remainder of one
          (1025, 8200, 1000),   # a strip of one row
          (2304, 8192, 200),    # 288 tiles: 256 whole, the other 32 in halves
          (2404, 8100, 300)]    # the same, and a strip of 100 rows behind the halves; ragged columns


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("kind", ["f16", "f32", "i32"])
def test_int8_weights(sess, oracle, M, N, K, kind):
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


@pytest.mark.parametrize("M,N,K", SHAPES)
@pytest.mark.parametrize("kind", ["f16", "f32", "i32", "swiglu"])
def test_int4_weights(sess, oracle, one_piece, M, N, K, kind):
    if kind == "swiglu":
        N = (N + 63) // 64 * 64
    c = workloads.w4a8_case(M, K, N, seed_w=N, seed_a=M)
    w = ops.W4A8Weights(sess, c["B"], c["w_scale"])
    ws = ops.W4A8Workspace(sess, M, N, K)
    try:
        A32 = oracle.half_to_float(c["A"]).astype(np.float32).reshape(M, K)
        if kind == "f16":
            (rc, got), kernels = one_piece(lambda: ws.run_f16(w, c["A"]))
            want = oracle.w4a8(c["A"], c["B"], c["w_scale"])["C"]
        elif kind == "f32":
            (rc, got), kernels = one_piece(lambda: ws.run_f32(w, A32))
            want = oracle.w4a8(A32, c["B"], c["w_scale"])["C"]
        elif kind == "i32":
            (rc, got), kernels = one_piece(lambda: ws.run_i32(w, A32))
            want = oracle.w4a8(A32, c["B"], c["w_scale"])["acc"]
        else:
            (rc, got), kernels = one_piece(lambda: ws.run_swiglu_f32(w, A32))
            want = oracle.w4a8_swiglu(A32, c["B"], c["w_scale"])["middle"]
        assert rc == 0 and kernels[-1] == "gemm_wk_big_kernel"
        assert np.array_equal(got.view(np.uint8), np.ascontiguousarray(want, got.dtype).view(np.uint8))
    finally:
        ws.close()
        w.close()


# A workgroup multiplies several 256 x 256 tiles as one stream of steps, then its share of the small ones: two and five trips of the
# loop per tile, three rounds with a last one of which some workgroups have no large tile
@pytest.mark.parametrize("M,N,K", [(4700, 8200, 512), (3000, 14336, 1100)])
@pytest.mark.parametrize("int4", [False, True])
def test_several_tiles_of_a_workgroup(sess, oracle, one_piece, M, N, K, int4):
    if int4:
        c = workloads.w4a8_case(M, K, N, seed_w=N, seed_a=M)
        w, ws = ops.W4A8Weights(sess, c["B"], c["w_scale"]), ops.W4A8Workspace(sess, M, N, K)
        (rc, got), kernels = one_piece(lambda: ws.run_f16(w, c["A"]))
        want = oracle.w4a8(c["A"], c["B"], c["w_scale"])["C"]
        ws.close()
        w.close()
    else:
        c = workloads.w8a8_case(M, K, N, seed_w=M, seed_a=K)
        op = ops.W8A8Linear(sess, capi.F16I8F16_DYNAMIC, M, c["B"], c["w_scale"])
        (rc, got), kernels = one_piece(lambda: op.run(c["A"]))
        want = oracle.w8a8(c["A"], c["B"], c["w_scale"])["C"]
        op.close()
    assert rc == 0 and kernels[-1] == "gemm_wk_big_kernel"
    assert np.array_equal(got.view(np.uint16), np.asarray(want).view(np.uint16))


# Small tiles behind a chain: (workgroups without a large tile in the last round, three small ones each; small ones on the others)
# 20 of 256 and 22, all of a last strip; 28 and 172, all halves of large tiles
@pytest.mark.parametrize("M,N,K,big,small,kind", [(1550, 20992, 512, 492, 82, kind) for kind in ("w8 f16", "w8 i32", "w4 f16", "w4 swiglu")] +
                         [(2968, 12951, 1024, 484, 256, kind) for kind in ("w8 f16", "w8 i32")])
def test_several_small_tiles_of_a_workgroup(sess, oracle, one_piece, M, N, K, big, small, kind):
    bits, kind = kind.split()
    v = [C.c_int() for _ in range(5)]
    epilogue = {"i32": 0, "f16": 1, "swiglu": 3}[kind]
    assert capi.load_library().rkh_gemm_route(M, N, K, int(bits == "w4"), epilogue, *[C.byref(x) for x in v]) == 0
    assert [x.value for x in v[1:]] == [256, 1, big, small]
    assert small > 3 * (256 - big % 256)  # (more than those without a large one take)
    if bits == "w4":
        c = workloads.w4a8_case(M, K, N, seed_w=N, seed_a=M)
        w, ws = ops.W4A8Weights(sess, c["B"], c["w_scale"]), ops.W4A8Workspace(sess, M, N, K)
        if kind == "f16":
            (rc, got), kernels = one_piece(lambda: ws.run_f16(w, c["A"]))
            want = oracle.w4a8(c["A"], c["B"], c["w_scale"])["C"]
        else:
            A32 = oracle.half_to_float(c["A"]).astype(np.float32).reshape(M, K)
            (rc, got), kernels = one_piece(lambda: ws.run_swiglu_f32(w, A32))
            want = oracle.w4a8_swiglu(A32, c["B"], c["w_scale"])["middle"]
        ws.close()
        w.close()
    else:
        c = workloads.w8a8_case(M, K, N, seed_w=M, seed_a=K)
        if kind == "f16":
            op, A = ops.W8A8Linear(sess, capi.F16I8F16_DYNAMIC, M, c["B"], c["w_scale"]), c["A"]
            want = oracle.w8a8(A, c["B"], c["w_scale"])["C"]
        else:
            A = np.random.default_rng(M).integers(-128, 128, (M, K)).astype(np.int8)
            op = ops.W8A8Linear(sess, capi.I8I8I32, M, c["B"])
            want = oracle.gemm_i8(A, c["B"])
        (rc, got), kernels = one_piece(lambda: op.run(A))
        op.close()
    assert rc == 0 and kernels[-1] == "gemm_wk_big_kernel"
    assert np.array_equal(got.view(np.uint8), np.ascontiguousarray(want, got.dtype).view(np.uint8))
