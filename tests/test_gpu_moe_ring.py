"""GPU parity of the balanced gate/up launch at its two ring depths (few or many units per compute unit), int8
experts, against the CPU oracle: K no multiple of 256, live row blocks far fewer than the call can have, the units per
compute unit on both sides of the line.  Exact.
"""
import numpy as np
import pytest

from rknpu2_matmul_open_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,H,I,E,top_k,one_expert,deep", [
    (13, 1056, 1024, 48, 4, False, True),   # 49 row blocks x 32 pairs: 6.1 units per compute unit
    (13, 1312, 1024, 52, 4, False, False),  # 53: 6.6
    (32, 1088, 1024, 44, 4, True, True),    # 48, of which four are live
    (13, 1024, 1024, 48, 4, False, False),  # the longest K that keeps the shallow ring
    (64, 1056, 512, 60, 3, False, True)])
def test_gate_up_ring(sess, oracle, T, H, I, E, top_k, one_expert, deep):
    rng = np.random.default_rng(T + H + E)
    experts = []
    for _ in range(E):
        experts.append((rng.integers(-127, 128, (H, 2 * I)).astype(np.int8), (rng.random(2 * I).astype(np.float32) + 0.5) * np.float32(0.02),
                        rng.integers(-127, 128, (I, H)).astype(np.int8), (rng.random(H).astype(np.float32) + 0.5) * np.float32(0.02)))
    x = rng.standard_normal((T, H)).astype(np.float32)
    ids = np.stack([np.arange(top_k) if one_expert else rng.permutation(E)[:top_k] for _ in range(T)]).astype(np.int32)
    routes = rng.random((T, top_k), dtype=np.float32) + np.float32(0.1)
    moe = ops.MoeW8(sess, H, I, E, 0, top_k, T, experts)
    dx, dids, drt = sess.to_device(x), sess.to_device(ids), sess.to_device(routes)
    dout = sess.empty_device(T * H * 4)
    try:
        rc2, want = oracle.moe_w8(experts, H, I, E, 0, top_k, ids, routes, input_f32=x)
        for _ in range(2):
            assert sess.lib.rk_npu_moe_w8_run_f32_device(moe.ws, moe.w, T, dx, dids, drt, dout) == 0 and sess.sync() == 0 and rc2 == 0
            got = sess.from_device(dout, (T, H), np.float32)
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        kernels = ops.profile_kernels(sess, lambda: sess.lib.rk_npu_moe_w8_run_f32_device(moe.ws, moe.w, T, dx, dids, drt, dout), 1, 0)
        assert kernels[1][0] == ("gemm_stream_kernel<balanced, four steps>" if deep else "gemm_stream_kernel<balanced>")
    finally:
        for d in (dx, dids, drt, dout):
            sess.free_device(d)
        moe.close()
