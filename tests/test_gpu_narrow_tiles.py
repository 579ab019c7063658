"""GPU parity of the 64 x 128 tiles of the LDS-ring GEMM on a long K (dense_narrow), against the CPU oracle.

The rule takes them by K and by the number of tiles; the cases stand at its edges (the fewest tiles of each
K range, and K just below and beyond a limit) with rows, columns and K that are no multiples of a tile.
Integer sums and a fixed order of the floating-point steps: exact.
"""
import numpy as np
import pytest

from rknpu2_matmul_open_amd import capi, ops, workloads

pytestmark = pytest.mark.gpu


# Row blocks x column blocks = 99 tiles (enough to K = 6656 int8 / 9728 int4), 129 (8192 / 13312), 162 (16384), 192 (24576, int4), and
# one K past a limit (K split)
@pytest.mark.parametrize("M,N,K", [(129, 4100, 6200), (129, 4100, 8500), (129, 5500, 8200), (129, 5500, 8100), (129, 6900, 8200)])
def test_int8_weights(sess, oracle, M, N, K):
    c = workloads.w8a8_case(M, K, N, seed_w=M, seed_a=K)
    op = ops.W8A8Linear(sess, capi.F16I8F16_DYNAMIC, M, c["B"], c["w_scale"])
    try:
        rc, got = op.run(c["A"])
        want = oracle.w8a8(c["A"], c["B"], c["w_scale"])["C"]
        assert rc == 0 and np.array_equal(got.view(np.uint16), np.asarray(want).view(np.uint16))
    finally:
        op.close()


@pytest.mark.parametrize("M,N,K", [(129, 4100, 11200), (129, 4100, 11300), (129, 5500, 11300), (129, 8100, 16400), (129, 4100, 8100),
                                   (129, 5500, 11200), (129, 5500, 13400), (129, 6900, 13400)])
def test_int4_weights(sess, oracle, M, N, K):
    c = workloads.w4a8_case(M, K, N, seed_w=N, seed_a=M)
    w = ops.W4A8Weights(sess, c["B"], c["w_scale"])
    ws = ops.W4A8Workspace(sess, M, N, K)
    try:
        rc, got = ws.run_f16(w, c["A"])
        want = oracle.w4a8(c["A"], c["B"], c["w_scale"])["C"]
        assert rc == 0 and np.array_equal(got.view(np.uint16), np.asarray(want).view(np.uint16))
    finally:
        ws.close()
        w.close()


@pytest.mark.parametrize("M,N,K", [(300, 2100, 40), (130, 4100, 512), (300, 3000, 1537), (320, 2900, 1792)])
def test_fewer_sub_steps_than_the_look_ahead(sess, oracle, M, N, K):
    """K of 2, 4, 14 (both) sub-steps where copies run twelve ahead: what is issued beyond K must not count."""
    c = workloads.w8a8_case(2, K, N, seed_w=M, seed_a=K)
    A = np.random.default_rng(K).integers(-128, 128, (M, K)).astype(np.int8)
    op = ops.W8A8Linear(sess, capi.I8I8I32, M, c["B"])
    try:
        rc, got = op.run(A)
        assert rc == 0 and np.array_equal(got, oracle.gemm_i8(A, c["B"]))
    finally:
        op.close()
