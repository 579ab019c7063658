"""What a user of this library has it do, as measurable cases.

Every case goes through the public C entry points as a program that links the
library calls them: the `*_device` calls with device pointers where
activations stay on the GPU between layers, the blocking reference calls with
host buffers where a program was only re-linked.  A case is one of

  linear   `layers` projections of one shape, one after the other, as a model
           runs the same projection of consecutive layers: per-token
           quantization, int8 or int4 weights, dequantized or exact result;
  ffn      `layers` gate/up + SwiGLU + down blocks on int4 weights
           (rk_npu_w4a8_run_ffn_f32*), the middle among the outputs;
  moe      one routed SwiGLU expert layer (rk_npu_moe_w8_run_f32*).

Several layers are used where few rows meet the weights (decode): each layer
has weights of its own, as in a model, so that they come from memory and not
from a cache that the previous call filled.

Results are compared exactly: the integer sums are exact in any order and the
floating-point steps around them (scale, two multiplies, SwiGLU polynomial,
ordered combine) are fixed by the interface, which promises the bits of the
reference's CPU path.
"""
import ctypes as C
import math

import numpy as np
import torch

from rknpu2_matmul_open_amd import capi, ops
from rknpu2_matmul_open_amd.capi import ptr

# What a linear call is named after: (input type, output type, bits of a weight).
_OPS = {
    "f16i8f16": (torch.float16, torch.float16, 8),
    "f32i8f32": (torch.float32, torch.float32, 8),
    "i8i8i32": (torch.int8, torch.int32, 8),
    "w4a8_f16": (torch.float16, torch.float16, 4),
    "w4a8_f32": (torch.float32, torch.float32, 4),
}
_W8_KIND = {"f16i8f16": capi.F16I8F16_DYNAMIC, "f32i8f32": capi.F32I8F32_DYNAMIC, "i8i8i32": capi.I8I8I32}
_BYTES = {torch.float16: 2, torch.float32: 4, torch.int8: 1, torch.int32: 4}

# The largest drawn case costs what the largest listed one does.
_MOST_PRODUCTS = 4096 * 4096 * 14336
_MOST_HOST_PRODUCTS = 2048 * 4096 * 4096


def _linear(name, op, M, K, N, layers=1, host=False):
    return {"name": name, "kind": "linear", "op": op, "M": M, "K": K, "N": N, "layers": layers, "host": host}


def _ffn(name, M, H, I, layers=1, host=False):
    return {"name": name, "kind": "ffn", "M": M, "H": H, "I": I, "layers": layers, "host": host}


def _moe(name, T, H, I, E, top_k, experts, host=False):
    return {"name": name, "kind": "moe", "T": T, "H": H, "I": I, "E": E, "top_k": top_k, "experts": experts, "host": host}


def listed():
    return [
        # One token of one sequence: the w8a8 decode projection of the benchmark (4096 -> 14336), four layers of it.
        _linear("decode_w8_1row", "f16i8f16", 1, 4096, 14336, layers=4),
        # One token through the int4 FFN block, two layers: the other half of a decode step.
        _ffn("decode_ffn_w4_1row", 1, 4096, 14336, layers=2),
        # Sixteen sequences decoded together: the down projection, where K is long and rows are few.
        _linear("batch16_w8_down", "f16i8f16", 16, 14336, 4096, layers=2),
        # A short prompt on a small model, fp32 activations, no size a multiple of anything: tails and latency.
        _linear("short_prompt_ragged", "f32i8f32", 61, 2050, 1999),
        # The exact int8 product of the reference's own benchmark at 128 rows (its ffn_up), device-resident.
        _linear("exact_i8_128rows", "i8i8i32", 128, 4096, 11008),
        # The int4 FFN block on a batch of 128 rows (many decoding sequences or a short prompt).
        _ffn("ffn_w4_128rows", 128, 4096, 14336),
        # The same block on a chunk of a prompt.
        _ffn("ffn_w4_512rows", 512, 4096, 14336),
        # Prefill: the w4a8 benchmark GEMM (2048 tokens, 4096 x 4096).
        _linear("prefill_w4_2048rows", "w4a8_f16", 2048, 4096, 4096),
        # A long prompt through the widest projection on int8 weights: the largest product.
        _linear("prefill_w8_4096rows", "f16i8f16", 4096, 4096, 14336),
        # The routed expert layer at its benchmark size: 256 tokens, 32 experts, top-4, int8 experts.
        _moe("moe_w8_256tokens", 256, 2048, 1024, 32, 4, "w8"),
        # The same layer while decoding: four tokens, int4 experts.
        _moe("moe_w4_4tokens", 4, 2048, 1024, 32, 4, "quant"),
        # A program that was only re-linked: the prefill GEMM on host buffers through the blocking call.
        _linear("host_prefill_w4_2048rows", "w4a8_f16", 2048, 4096, 4096, host=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, step):
    """A size of lo..hi: mostly a multiple of `step`, now and then any number."""
    v = _log_int(rng, lo, hi)
    if rng.random() < 0.3:
        return v
    return max(lo // step, round(v / step)) * step


def _layers(rows, weight_bytes):
    """Layers of a drawn case: few rows meet weights that come from memory (up to eight layers, about 128 MB)."""
    return 1 if rows > 64 else max(1, min(8, int(128e6 / weight_bytes)))


def draw(rng):
    kind = rng.choice(["linear"] * 5 + ["ffn"] * 2 + ["moe"] * 2 + ["host"])
    if kind == "linear" or kind == "host":
        host = kind == "host"
        most = _MOST_HOST_PRODUCTS if host else _MOST_PRODUCTS
        while True:
            M = _log_int(rng, 1, 2048 if host else 4096)
            K, N = _size(rng, 512, 14336, 128), _size(rng, 512, 14336, 128)
            if M * K * N <= most:
                break
        op = rng.choice(sorted(_OPS))
        return _linear_drawn(op, M, K, N, _layers(M, K * N * _OPS[op][2] // 8), host)
    if kind == "ffn":
        while True:
            M = _log_int(rng, 1, 2048)
            H, I = _log_int(rng, 512, 5120) // 32 * 32, _log_int(rng, 1024, 14336) // 32 * 32
            if 3 * M * H * I <= _MOST_PRODUCTS:
                break
        return {"kind": "ffn", "M": M, "H": H, "I": I, "layers": _layers(M, 3 * H * I // 2), "host": False}
    while True:
        H, I = _log_int(rng, 512, 4096) // 64 * 64, _log_int(rng, 256, 2048) // 64 * 64
        E = _log_int(rng, 8, 64)
        if 3 * H * I * E <= 3 * 2048 * 1024 * 32:
            break
    return {"kind": "moe", "T": _log_int(rng, 1, 256), "H": H, "I": I, "E": E, "top_k": rng.randint(1, 8),
            "experts": rng.choice(["w8", "quant"]), "host": False}


def _linear_drawn(op, M, K, N, layers, host):
    return {"kind": "linear", "op": op, "M": M, "K": K, "N": N, "layers": layers, "host": host}


def work(case):
    if case["kind"] == "linear":
        M, K, N = case["M"], case["K"], case["N"]
        a, c, bits = _OPS[case["op"]]
        one = M * K * _BYTES[a] + M * N * _BYTES[c] + K * N * bits // 8 + (4 * N if case["op"] != "i8i8i32" else 0)
        return {"bytes": case["layers"] * one, "flops": case["layers"] * 2 * M * K * N}
    if case["kind"] == "ffn":
        M, H, I = case["M"], case["H"], case["I"]
        one = 3 * H * I // 2 + 4 * (2 * I + H) + 4 * M * (H + I + H)  # weights, scales, input, middle, output
        return {"bytes": case["layers"] * one, "flops": case["layers"] * 6 * M * H * I}
    T, H, I, E, k = case["T"], case["H"], case["I"], case["E"], case["top_k"]
    met = E * (1.0 - (1.0 - k / E) ** T)  # experts that some token is routed to, on average
    expert = 3 * H * I // (1 if case["experts"] == "w8" else 2) + 4 * (2 * I + H)
    return {"bytes": met * expert + T * (8 * H + 8 * k), "flops": 6.0 * T * k * H * I}


def tolerance(case):
    return "exact"


# ---- what a program holds before the call --------------------------------------------------

_sessions = []


def _session():
    """The process's one context and domain, as a program opens them once."""
    if not _sessions:
        _sessions.append(ops.Session())
    return _sessions[0]


class _Held:
    """A case's handles and buffers; the handles are given back with the object."""

    def __init__(self):
        self.handles, self.calls, self.outputs, self.buffers = [], [], [], []

    def __del__(self):
        for h in self.handles:
            h.close()


def _quantized_weight(gen, K, N, qmax):
    """N(0, 0.02) weights of a projection, quantized per output channel: codes [K, N] and scales [N] on the host."""
    w = torch.randn((K, N), generator=gen, device="cuda").mul_(0.02)
    scale = w.abs().amax(dim=0).clamp_(min=1e-12) / qmax
    codes = torch.round(w / scale).clamp_(-qmax, qmax).to(torch.int8)
    return codes.cpu().numpy(), scale.cpu().numpy()


def _activations(gen, M, K, dtype):
    """N(0, 1) rows with the outliers that activations show (0.5 % of the values, twenty times larger)."""
    if dtype is torch.int8:
        return torch.round(torch.randn((M, K), generator=gen, device="cuda") * 32).clamp_(-127, 127).to(torch.int8)
    x = torch.randn((M, K), generator=gen, device="cuda")
    far = torch.rand((M, K), generator=gen, device="cuda") < 0.005
    return torch.where(far, x * 20, x).to(dtype)


def _buffer(held, tensor, host):
    """The tensor where the call takes it from (or writes it to), and its address."""
    if host:
        array = np.array(tensor.cpu().numpy())
        held.buffers.append(array)
        return array, ptr(array)
    held.buffers.append(tensor)
    return tensor, C.c_void_p(tensor.data_ptr())


def _prepare_linear(case, gen, held):
    s = _session()
    lib, host = s.lib, case["host"]
    M, K, N, op = case["M"], case["K"], case["N"], case["op"]
    a_type, c_type, bits = _OPS[op]
    shared = None
    for _ in range(case["layers"]):
        codes, scale = _quantized_weight(gen, K, N, 127 if bits == 8 else 7)
        _, a = _buffer(held, _activations(gen, M, K, a_type), host)
        out, c = _buffer(held, torch.zeros((M, N), dtype=c_type, device="cuda"), host)
        held.outputs.append(out)
        if bits == 8:
            # (one workspace per layer: the wrapper creates both)
            lin = ops.W8A8Linear(s, _W8_KIND[op], M, codes, None if op == "i8i8i32" else scale)
            held.handles.append(lin)
            name = {"f16i8f16": "rk_npu_f16i8f16_run_dynamic", "f32i8f32": "rk_npu_f32i8f32_run_dynamic",
                    "i8i8i32": "rk_npu_i8i8i32_run"}[op] + ("" if host else "_device")
            held.calls.append((getattr(lib, name), (lin.ws, lin.w, a, c)))
        else:
            w = ops.W4A8Weights(s, codes, scale)
            if shared is None:  # one workspace serves every layer of a shape
                shared = ops.W4A8Workspace(s, M, N, K)
                held.handles.append(shared)
            held.handles.append(w)
            name = "rk_npu_w4a8_run_" + op[-3:] + ("" if host else "_device")
            held.calls.append((getattr(lib, name), (shared.h, w.h, a, c) + ((None,) if host else ())))


def _prepare_ffn(case, gen, held):
    s = _session()
    M, H, I, host = case["M"], case["H"], case["I"], case["host"]
    gu_ws, dn_ws = ops.W4A8Workspace(s, M, 2 * I, H), ops.W4A8Workspace(s, M, H, I)
    held.handles += [gu_ws, dn_ws]
    for _ in range(case["layers"]):
        gu = ops.W4A8Weights(s, *_quantized_weight(gen, H, 2 * I, 7))
        dn = ops.W4A8Weights(s, *_quantized_weight(gen, I, H, 7))
        held.handles += [gu, dn]
        _, a = _buffer(held, _activations(gen, M, H, torch.float32), host)
        middle, m = _buffer(held, torch.zeros((M, I), device="cuda"), host)
        out, c = _buffer(held, torch.zeros((M, H), device="cuda"), host)
        held.outputs += [middle, out]
        fn = s.lib.rk_npu_w4a8_run_ffn_f32 if host else s.lib.rk_npu_w4a8_run_ffn_f32_device
        held.calls.append((fn, (gu_ws.h, gu.h, dn_ws.h, dn.h, a, m, c) + ((None,) if host else ())))


def _prepare_moe(case, gen, held):
    s = _session()
    T, H, I, E, k, host = case["T"], case["H"], case["I"], case["E"], case["top_k"], case["host"]
    qmax = 127 if case["experts"] == "w8" else 7
    experts = []
    for _ in range(E):
        gate_up, gate_up_scale = _quantized_weight(gen, H, 2 * I, qmax)
        down, down_scale = _quantized_weight(gen, I, H, qmax)
        experts.append((gate_up, gate_up_scale, down, down_scale))
    layer = ops.MoeW8(s, H, I, E, 0, k, T, experts, flavour=case["experts"])
    held.handles.append(layer)
    p = torch.softmax(torch.randn((T, E), generator=gen, device="cuda"), dim=1)
    p, ids = torch.topk(p, k, dim=1)
    _, x = _buffer(held, _activations(gen, T, H, torch.float32), host)
    _, ids = _buffer(held, ids.to(torch.int32).contiguous(), host)
    _, routes = _buffer(held, (p / p.sum(dim=1, keepdim=True)).contiguous(), host)
    out, c = _buffer(held, torch.zeros((T, H), device="cuda"), host)
    held.outputs.append(out)
    fn = s.lib.rk_npu_moe_w8_run_f32 if host else s.lib.rk_npu_moe_w8_run_f32_device
    held.calls.append((fn, (layer.ws, layer.w, T, x, ids, routes, c) + ((None,) if host else ())))


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    held = _Held()
    {"linear": _prepare_linear, "ffn": _prepare_ffn, "moe": _prepare_moe}[case["kind"]](case, gen, held)
    torch.cuda.synchronize()
    return held


def run(state):
    for fn, args in state.calls:
        rc = fn(*args)
        if rc:
            raise ops.RkError(rc, "pass")
    return state.outputs
