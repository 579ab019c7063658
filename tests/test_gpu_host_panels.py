"""GPU parity of large blocking calls on host buffers, which go in panels of rows, against the CPU oracle.

A and C are just large enough for panels (tests/host_calls_cpu.cpp holds which calls are); the panels are 128 rows and the last one is whole, one row (the decode
kernel), a few rows or nearly whole.  Also: the quantized rows that the call leaves in its workspace, given scales,
rejected input in the first and the last panel or in an earlier device call (C stays as it was) and two threads at once.
Exact.
"""
import threading

import numpy as np
import pytest

from rknpu2_matmul_open_amd import capi, ops, workloads

pytestmark = pytest.mark.gpu

K, N = 2850, 4224  # 128 rows of fp32 results: 2.1 MiB, the size of a panel


@pytest.mark.parametrize("M", [384, 385, 389, 510])
@pytest.mark.parametrize("kind", ["dynamic", "static", "i32"])
def test_int8_weights(sess, oracle, M, kind):
    c = workloads.w8a8_case(2, K, N, seed_w=M, seed_a=1)
    scale = None
    if kind == "i32":
        A = np.random.default_rng(M).integers(-128, 128, (M, 4 * K)).astype(np.int8)  # (more than 4 MiB)
        B = np.concatenate([c["B"], c["B"][::-1], c["B"][:, ::-1], c["B"]])
        op, want = ops.W8A8Linear(sess, capi.I8I8I32, M, B), oracle.gemm_i8(A, B)
    else:
        A = workloads.normal_f32(M, (M, K))
        scale = (np.abs(A).max(axis=1) / 100).astype(np.float32) if kind == "static" else None
        op = ops.W8A8Linear(sess, capi.F32I8F32_STATIC if kind == "static" else capi.F32I8F32_DYNAMIC, M, c["B"], c["w_scale"])
        full = oracle.w8a8(A, c["B"], c["w_scale"], scale)
        want = full["C"]
    try:
        for _ in range(2):
            rc, got = op.run(A, scale)
            assert rc == 0
            assert np.array_equal(got.view(np.uint32), np.ascontiguousarray(want).view(np.uint32))
        if kind != "i32":
            q, s = op.read_quantized()
            assert np.array_equal(q, full["q"]) and np.array_equal(s, full["a_scale"])
    finally:
        op.close()


@pytest.mark.parametrize("M", [384, 387, 510])
def test_int4_weights(sess, oracle, M):
    c = workloads.w4a8_case(M, K, N, seed_w=5, seed_a=M)
    A = oracle.half_to_float(c["A"]).astype(np.float32).reshape(M, K)
    w, ws = ops.W4A8Weights(sess, c["B"], c["w_scale"]), ops.W4A8Workspace(sess, M, N, K)
    want = oracle.w4a8(A, c["B"], c["w_scale"])["C"]
    try:
        rc, got = ws.run_f32(w, A)
        assert rc == 0 and np.array_equal(got.view(np.uint32), want.view(np.uint32))
        for row in (3, M - 1):
            bad, C = A.copy(), np.full((M, N), 7.0, np.float32)
            bad[row, K - 1] = np.inf
            assert sess.lib.rk_npu_w4a8_run_f32(ws.h, w.h, capi.ptr(bad), capi.ptr(C), None) == capi.RK_NPU_ERR_PARAM
            assert np.all(C == 7.0)
        rc, got = ws.run_f32(w, A)
        assert rc == 0 and np.array_equal(got.view(np.uint32), want.view(np.uint32))
    finally:
        ws.close()
        w.close()


def test_an_earlier_device_call_rejected_its_input(sess, oracle):
    """... and nothing has synchronized since: the blocking call says so and leaves C alone, the next one is good."""
    M = 389
    c = workloads.w4a8_case(M, K, N, seed_w=5, seed_a=M)
    A = oracle.half_to_float(c["A"]).astype(np.float32).reshape(M, K)
    bad = A.copy()
    bad[M - 1, 0] = np.nan
    w, ws = ops.W4A8Weights(sess, c["B"], c["w_scale"]), ops.W4A8Workspace(sess, M, N, K)
    dA, dC, C = sess.to_device(bad), sess.empty_device(M * N * 4), np.full((M, N), 7.0, np.float32)
    try:
        assert sess.lib.rk_npu_w4a8_run_f32_device(ws.h, w.h, dA, dC) == 0
        assert sess.lib.rk_npu_w4a8_run_f32(ws.h, w.h, capi.ptr(A), capi.ptr(C), None) == capi.RK_NPU_ERR_PARAM
        assert np.all(C == 7.0)
        rc, got = ws.run_f32(w, A)
        assert rc == 0 and np.array_equal(got.view(np.uint32), oracle.w4a8(A, c["B"], c["w_scale"])["C"].view(np.uint32))
        assert sess.sync() == 0
    finally:
        sess.free_device(dA)
        sess.free_device(dC)
        ws.close()
        w.close()


def test_two_threads(sess, oracle):
    M = 389
    c = workloads.w8a8_case(2, K, N, seed_w=9, seed_a=1)
    lin = [ops.W8A8Linear(sess, capi.F32I8F32_DYNAMIC, M, c["B"], c["w_scale"]) for _ in range(2)]
    As = [workloads.normal_f32(70 + i, (M, K)) for i in range(2)]
    wants = [oracle.w8a8(A, c["B"], c["w_scale"])["C"] for A in As]
    errors = []

    def work(i):
        for it in range(6):
            rc, got = lin[i].run(As[i])
            if rc or not np.array_equal(got.view(np.uint32), wants[i].view(np.uint32)):
                errors.append((i, it, rc))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    try:
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not errors, errors
    finally:
        for op in lin:
            op.close()


def test_a_profile_sees_every_kernel(sess, oracle):
    """While a per-kernel profile is on, which marks the context's stream, the call runs on it in one piece."""
    import ctypes as C
    M = 389
    c = workloads.w8a8_case(2, K, N, seed_w=3, seed_a=1)
    A = workloads.normal_f32(5, (M, K))
    op = ops.W8A8Linear(sess, capi.F32I8F32_DYNAMIC, M, c["B"], c["w_scale"])
    buf, us = C.create_string_buffer(4096), (C.c_double * 16)()
    try:
        assert sess.lib.rk_npu_hip_profile_begin(sess.ctx) == 0
        rc, got = op.run(A)
        n = sess.lib.rk_npu_hip_profile_end(sess.ctx, buf, len(buf), us, 16)
        assert rc == 0 and 2 <= n <= 3  # quantization, GEMM and, if its K is split, the sum of the parts
        assert np.array_equal(got.view(np.uint32), oracle.w8a8(A, c["B"], c["w_scale"])["C"].view(np.uint32))
    finally:
        op.close()
