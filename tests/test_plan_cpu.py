"""Host logic of the dense launch plan, through the one function of it the library exports for sizing
a workspace: the bytes of split-K scratch, = tiles x K split x tile rows x 256 columns x 4.  No GPU call
is made (the plan is arithmetic on the shape)."""
import ctypes as C
import json
import os
import subprocess
import sys

import pytest

from rknpu2_matmul_open_amd import capi


@pytest.fixture(scope="module")
def scratch_bytes():
    lib = capi.load_library()
    f = lib.rkh_gemm_scratch_bytes
    f.restype = C.c_size_t
    f.argtypes = [C.c_int] * 4
    return f


def _ksplit(nbytes, M, N):
    """K split implied by the scratch size (rows are padded to the tile, so try every tile height)."""
    found = set()
    for bm in (128, 64, 32):
        tiles = -(-M // bm) * -(-N // 256)
        per_part = tiles * bm * 256 * 4
        if nbytes % per_part == 0:
            found.add(nbytes // per_part)
    return found


# (M, N, K, int4) -> K split the plan chooses; the choices measured fastest (or within a few percent of it)
# among forced plans on the device: long K with few columns is split, wide or short-K GEMMs are not
PINNED = [((192, 4096, 4096, 0), 4), ((256, 4096, 4096, 0), 4), ((512, 4096, 4096, 0), 0), ((1024, 4096, 4096, 0), 0),
          ((192, 11008, 4096, 0), 0), ((512, 11008, 4096, 0), 0), ((1024, 14336, 4096, 0), 0),
          ((192, 4096, 11008, 0), 4), ((256, 4096, 11008, 0), 4), ((512, 4096, 11008, 0), 4), ((1024, 4096, 11008, 0), 2),
          ((2048, 4096, 4096, 1), 0), ((2048, 4096, 4096, 0), 0), ((512, 4096, 11008, 1), 2), ((192, 4096, 4096, 1), 0)]


@pytest.mark.parametrize("shape,ksplit", PINNED)
def test_k_split_of_measured_shapes(scratch_bytes, shape, ksplit):
    M, N, K, int4 = shape
    nbytes = scratch_bytes(M, N, K, int4)
    if ksplit == 0:
        assert nbytes == 0
    else:
        assert ksplit in _ksplit(nbytes, M, N), (nbytes, _ksplit(nbytes, M, N))


def test_plan_invariants(scratch_bytes):
    # decode-sized calls never split over workgroups
    for M in range(1, 9):
        assert scratch_bytes(M, 4096, 14336, 0) == 0 and scratch_bytes(M, 4096, 14336, 1) == 0
    # int4 weights ride as 16 x code: a part may not span more than 2^17 k, whatever the estimate prefers
    for M in (200, 2000):
        nbytes = scratch_bytes(M, 96, 131072 + 2112, 1)
        assert nbytes > 0 and min(_ksplit(nbytes, M, 96)) >= 2
        nbytes = scratch_bytes(M, 96, 3 * 131072 + 64, 1)
        assert nbytes > 0 and min(_ksplit(nbytes, M, 96)) >= 4
    # a part keeps at least 1024 k, and the scratch stays bounded
    assert scratch_bytes(4000, 256, 1500, 0) == 0
    for shape in ((300001, 300, 33, 0), (100000, 256, 8192, 0), (5000, 64, 60000, 0), (129, 3000001, 40, 0)):
        assert scratch_bytes(*shape) <= 512 * 1000 * 1000


def test_which_moe_calls_take_the_two_launch_path():
    """Up to twelve tokens, a hidden size that fits the staging area, a middle short enough for nine
    re-quantized rows side by side; everything else takes the routed, grouped path."""
    lib = capi.load_library()
    f = lib.rkh_moe_decode_applies
    f.restype = C.c_int
    f.argtypes = [C.c_int] * 3
    for rows in range(1, 13):
        assert f(rows, 2048, 1024) and f(rows, 64, 32) and f(rows, 32768, 3584)
    assert not f(13, 2048, 1024) and not f(256, 2048, 1024) and not f(0, 2048, 1024)
    assert not f(4, 32768 + 32, 1024) and not f(4, 2048, 3584 + 32) and not f(4, 2048, 8192)
    assert not f(4, 2040, 1024) and not f(4, 2048, 1000)   # (the layer's geometry is in multiples of 32)


# ---- which kernel a dense call takes (the same rules rkh_gemm applies) ----
FEW, GEMV, GEMV_SWIGLU, STREAM, TILES_NARROW, TILES = range(6)
EPI_I32, EPI_F16, EPI_F32, EPI_SWIGLU = range(4)


@pytest.fixture(scope="module")
def route():
    lib = capi.load_library()
    f = lib.rkh_gemm_route
    f.restype = C.c_int
    f.argtypes = [C.c_int] * 5 + [C.POINTER(C.c_int)] * 5

    def call(M, N, K, int4=0, epilogue=EPI_F16, cut=False):
        out = [C.c_int(-1) for _ in range(5)]
        assert f(M, N, K, int4, epilogue, *[C.byref(v) for v in out]) == 0
        return tuple(v.value for v in out)[3 if cut else 0:5 if cut else 3]
    return call


@pytest.mark.parametrize("epilogue", [EPI_I32, EPI_F16, EPI_F32])
def test_few_rows_of_a_k_beyond_a_descriptor(route, epilogue):
    """gemm_few_kernel addresses a column block over all of K, 32 K bytes, through a 32-bit descriptor: from
    K = 2^27 on its loads would return zeros.  The streaming kernel, whose strides are 64-bit, keeps such rows."""
    for M in (9, 16, 17, 32, 40, 64):
        for K in ((1 << 26) - 200, 1 << 26, 1 << 27, (1 << 27) + 256, (1 << 31) - 257):
            for N in (1, 256, 5000):
                assert route(M, N, K, 0, epilogue)[0] == STREAM, (M, N, K)
    assert route(16, 4096, 14336, 0, epilogue) == (FEW, 16, 1)
    # int4 weights ride as 16 x code in an int32 sum
    for M in (9, 16, 32):
        assert route(M, 256, 131072 + 256, 1, epilogue)[0] not in (FEW, STREAM)


@pytest.mark.parametrize("epilogue", [EPI_I32, EPI_F16, EPI_F32])
def test_decode_rows_of_a_k_beyond_a_descriptor(route, epilogue):
    """The same 32-bit descriptor in the decode kernel: 32 K bytes of int8 weights have to be less than 2^32."""
    for M in range(1, 9):
        for K in (1 << 27, (1 << 27) - 255, (1 << 27) + 256, (1 << 31) - 257):
            for N in (1, 256, 5000):
                assert route(M, N, K, 0, epilogue)[0] == STREAM, (M, N, K)
        assert route(M, 256, (1 << 27) - 256, 0, epilogue)[0] == GEMV


_ROUTES = """
import ctypes as C, json, sys
from rknpu2_matmul_open_amd import capi
f = capi.load_library().rkh_gemm_route
got = []
for shape in json.loads(sys.argv[1]):
    out = [C.c_int(-1) for _ in range(5)]
    assert f(*[C.c_int(v) for v in shape], *[C.byref(v) for v in out]) == 0
    got.append([v.value for v in out[:3]])
print(json.dumps(got))
"""


def _routes_under(env, shapes):
    """Routes with environment switches set (the library reads them once per process)."""
    child = subprocess.run([sys.executable, "-c", _ROUTES, json.dumps(shapes)], env=dict(os.environ, **env), text=True,
                           capture_output=True, timeout=120, cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    assert child.returncode == 0, child.stderr[-2000:]
    return [tuple(r) for r in json.loads(child.stdout.strip().splitlines()[-1])]


def test_forced_256_row_tiles_never_drop_a_k_split():
    """256 x 256 tiles walk all of K in one accumulator: forced for int4 weights of more than 2^17 k, whose sums
    of 16 x code may wrap, or with a split, they are no plan and the computed one stays."""
    shapes = [[2000, 4096, 4096, 0, EPI_F16], [300, 512, 131072, 1, EPI_F32], [300, 512, 131072 + 256, 1, EPI_F32],
              [2000, 4096, 3 * 131072, 1, EPI_F16]]
    got = _routes_under({"RK_NPU_HIP_GEMM_PLAN": "256:1"}, shapes)
    assert got[:2] == [(TILES, 256, 1)] * 2
    for kernel, rows, ksplit in got[2:]:
        assert kernel == TILES and rows <= 128 and ksplit >= 2
    free = _routes_under({"RK_NPU_HIP_GEMM_PLAN": "none"}, shapes)  # (no plan, but read as a forced one: no other rule)
    assert got[2:] == free[2:]
    assert _routes_under({"RK_NPU_HIP_GEMM_PLAN": "256:2"}, shapes) == free


def test_forced_kernels_take_their_rows():
    """The switches that force a width or a row limit of the decode or the streaming kernel: gemm_few_kernel, which
    takes rows of both by default, leaves these calls to them."""
    decode = [[5, 72, 20000, 0, EPI_F16], [8, 300, 8192, 0, EPI_I32], [4, 72, 140000, 1, EPI_F16]]
    more = [[16, 4096, 4096, 0, EPI_F16], [64, 8192, 4096, 0, EPI_F32], [16, 4096, 4096, 1, EPI_F16]]
    assert [r[0] for r in _routes_under({}, decode + more)] == [FEW, FEW, GEMV, FEW, FEW, FEW]
    for switch in ({"RK_NPU_HIP_GEMV_COLS": "16"}, {"RK_NPU_HIP_GEMV_MAX_ROWS": "8"}):
        assert [r[0] for r in _routes_under(switch, decode + more)] == [GEMV] * 3 + [FEW] * 3
    got = _routes_under({"RK_NPU_HIP_GEMV_MAX_ROWS": "2"}, decode[:2] + [[2, 72, 20000, 0, EPI_F16]])
    assert [r[0] for r in got] == [STREAM, STREAM, GEMV]
    assert [r[0] for r in _routes_under({"RK_NPU_HIP_STREAM_MAX_ROWS": "128"}, decode + more)] == [GEMV] * 3 + [STREAM] * 3


def test_where_few_rows_keep_the_streaming_or_decode_kernel(route):
    """int8 weights: shapes among those gemm_few_kernel is best for at which it measured slower than the kernel that
    had them, and their neighbours on its side."""
    def kernel(M, N, K):
        return route(M, N, K)[0]
    for M, N, K in ((16, 4128, 2304), (32, 5120, 2300), (16, 9216, 2304), (9, 12288, 2560), (16, 28672, 2304), (16, 9216, 4608),
                    (9, 20480, 512), (16, 28672, 1024), (16, 8320, 8192), (12, 13312, 8192), (9, 28672, 8192),
                    (40, 4128, 2048), (64, 5120, 2048), (56, 6144, 1536), (64, 7168, 2048),
                    (33, 8320, 3072), (40, 8448, 5120), (56, 8320, 8192), (56, 9216, 8192), (56, 9216, 2048), (33, 9216, 1024), (57, 12288, 4096)):
        assert kernel(M, N, K) == STREAM, (M, N, K)
    for M, N, K in ((16, 4096, 2304), (16, 8192, 2304), (32, 4128, 2048), (16, 4128, 2560), (16, 20480, 2560), (16, 9216, 2816), (16, 12288, 4608),
                    (9, 14336, 512), (16, 20480, 1024), (16, 8192, 8192), (16, 20480, 8192), (16, 32768, 8192),
                    (64, 4128, 1024), (40, 5120, 2048), (48, 7168, 2048), (64, 8192, 2048), (64, 4128, 2560),
                    (56, 8512, 3072), (48, 9216, 8192), (40, 9216, 2048), (56, 14336, 14336)):
        assert kernel(M, N, K) == FEW, (M, N, K)
    assert [kernel(M, 14336, 8192) for M in (5, 6, 7, 8)] == [GEMV, GEMV, FEW, FEW] and kernel(5, 12288, 8192) == FEW


def test_64_row_tiles_of_a_long_k_run_in_one_round(route):
    """Three row blocks of an 11008-wide matrix are 258 tiles of 64 x 128: on 256 compute units a second round of
    two, which K <= 6144 tolerates and a longer K does not (the 128 x 128 tiles take it, whatever K)."""
    for M in (129, 160, 192):
        for K in (6145, 6400, 8192, 11008, 16384, 16385, 20480, 28672):
            assert route(M, 11008, K) == (TILES_NARROW, 128, 1), (M, K)
        for K in (2000, 6144):
            assert route(M, 11008, K) == (TILES_NARROW, 64, 1), (M, K)
        assert route(M, 10752, 8192) == (TILES_NARROW, 64, 1) and route(M, 10880, 14336) == (TILES_NARROW, 64, 1)
        assert route(M, 10752, 28672) == (TILES_NARROW, 128, 1)   # (no number of tiles pays beyond K = 16384)
        assert route(M, 11008, 8192, 1)[0] == TILES               # (int4 weights: no tiles of 128 x 128)


def test_fewest_64_row_tiles_of_a_long_k(route):
    """Fewer tiles, each walking its K alone, are slower than the K split once the weights come from memory."""
    for int4, K, least in ((0, 6656, 96), (0, 6657, 112), (0, 8192, 112), (0, 8193, 160), (0, 16384, 160),
                           (1, 9728, 96), (1, 9729, 112), (1, 11264, 112), (1, 11265, 128), (1, 13312, 128), (1, 13313, 160),
                           (1, 16384, 160), (1, 16385, 192), (1, 24576, 192), (1, 24577, 224), (1, 32768, 224)):
        for tiles in (least - 4, least, 252):                # four row blocks x a quarter of the tiles
            kernel, rows, ksplit = route(256, tiles // 4 * 128, K, int4)
            if tiles >= least:
                assert (kernel, rows, ksplit) == (TILES_NARROW, 64, 1), (int4, K, tiles)
            else:
                assert kernel == TILES, (int4, K, tiles)


@pytest.mark.parametrize("int4", [0, 1])
def test_cut_of_the_large_tiles(route, int4):
    """How a launch is cut into 256 x 256 tiles and 128 x 256 ones -- halves of the last 256 x 256 tiles, then a last
    strip of at most 128 rows; the shapes are those of test_gpu_large_tiles.py, which rely on it."""
    for M, N, K, big, halves, strip in ((1100, 7500, 200, 120, 0, 30), (1224, 7457, 300, 150, 0, 0), (2816, 6656, 513, 286, 0, 0),
                                        (1025, 8200, 1000, 132, 0, 33), (2304, 8192, 200, 256, 64, 0), (2404, 8100, 300, 256, 64, 32)):
        assert route(M, N, K, int4) == (TILES, 256, 1), (M, N, K)
        assert route(M, N, K, int4, cut=True) == (big, halves + strip), (M, N, K)
    assert route(4096, 14336, 4096, int4, cut=True) == (768, 256)
    assert route(2048, 4096, 4096, int4, cut=True) == (0, 0)


# ---- which rows the workgroups of a quantization launch take ----
Q_W8_DYNAMIC, Q_W4A8, Q_COPY_I8, Q_REUSE, Q_REUSE_MOE = 0, 2, 4, 5, 6
F16, F32, I8 = 0, 1, 2
DIES = 8  # workgroup b of a launch runs on die b % 8


class _QuantArgs(C.Structure):
    _fields_ = [("src", C.c_void_p), ("in_dtype", C.c_int), ("mode", C.c_int), ("M", C.c_int), ("K", C.c_int),
                ("scale", C.c_void_p), ("dst", C.c_void_p), ("bad_flag", C.c_void_p), ("row_max_bits", C.c_void_p),
                ("row_max_parts", C.c_int), ("active_blocks", C.c_void_p), ("src_is_host", C.c_int)]


@pytest.fixture(scope="module")
def dealing():
    f = capi.load_library().rkh_quant_row_of
    f.restype = C.c_int
    f.argtypes = [C.POINTER(_QuantArgs), C.c_int, C.c_int] + [C.POINTER(C.c_int)] * 3

    def call(M, K, dtype, mode, grouped=False, ahead=True):
        """[(die, first row, rows, part)] of every workgroup (grouped: only the first rows are live; ahead: of a GEMM,
        as nearly all of them are)"""
        a = _QuantArgs(in_dtype=dtype, mode=mode, M=M, K=K, row_max_parts=K // 32, active_blocks=1 if grouped else None)
        n, rows, part = C.c_int(1), C.c_int(0), C.c_int(0)
        got, b = [], 0
        while b < n.value:
            first = f(C.byref(a), int(ahead), b, C.byref(n), C.byref(rows), C.byref(part))
            got.append((b % DIES, first, rows.value, part.value))
            b += 1
        return got
    return call


@pytest.mark.parametrize("M", [1, 2, 7, 8, 9, 31, 32, 33, 61, 63, 64, 65, 100, 128, 255, 256, 257, 700, 767, 768, 1025, 4099])
@pytest.mark.parametrize("ahead", [False, True])
def test_every_row_is_quantized_once(dealing, M, ahead):
    for K in (40, 1024, 2048, 4096, 4128, 8224, 14336, 20000):
        for dtype, mode, grouped in ((F16, Q_W8_DYNAMIC, False), (F32, Q_W4A8, False), (I8, Q_COPY_I8, False),
                                     (F32, Q_REUSE, False), (F32, Q_REUSE_MOE, True)):
            seen = {}
            for _, first, rows, part in dealing(M, K, dtype, mode, grouped, ahead):
                assert first >= 0
                for row in range(first, min(first + rows, M)):
                    assert (row, part) not in seen
                    seen[row, part] = True
            parts = 1 + max(part for _, part in seen)
            # (scanned rows are shared only ahead of a GEMM, and only where the parts' registers hold a whole row)
            scanned = ahead and mode in (Q_W8_DYNAMIC, Q_W4A8) and 4096 < K <= 16384
            assert len(seen) == M * parts and (parts == 1 or mode in (Q_REUSE, Q_REUSE_MOE) or scanned), (K, dtype, mode)


@pytest.mark.parametrize("M,K,dtype,parts", [
    (1, 4096, F16, 1), (1, 4097, F16, 2), (128, 4104, F16, 2), (129, 4104, F16, 1), (128, 8192, F32, 2), (129, 8192, F32, 1),
    (1, 8200, F16, 4), (64, 8200, F16, 4), (128, 8200, F16, 4), (129, 8200, F16, 1), (128, 16384, F32, 4), (128, 16400, F32, 1),
    (64, 9001, F32, 4), (65, 9001, F32, 1), (64, 9001, F16, 4), (65, 9001, F16, 1), (128, 8196, F32, 4), (65, 8196, F16, 1)])
def test_workgroups_that_share_a_scanned_row(dealing, M, K, dtype, parts):
    """Two up to 8192 elements, four up to 16384, while that makes 256 workgroups at most, or 512 of rows whose chunks are
    16-byte aligned and that four share; each part once, the parts of a row in consecutive places of one die's range."""
    for mode in (Q_W8_DYNAMIC, Q_W4A8):
        got = dealing(M, K, dtype, mode)
        assert sorted((row, part) for _, row, _, part in got) == [(m, p) for m in range(M) for p in range(parts)]
        assert len(dealing(M, K, dtype, mode, ahead=False)) == M
        if parts > 1:
            for die in range(DIES):
                mine = [row * parts + part for d, row, _, part in got if d == die]
                assert not mine or mine == list(range(mine[0], mine[0] + len(mine)))


@pytest.mark.parametrize("I", [512, 1024, 4096, 4128, 8224])
def test_live_rows_of_a_moe_call_are_spread_over_the_dies(dealing, I):
    """A workspace holds more row blocks than a call fills, and the live ones are the first: whatever their
    number, the dies' shares differ by a group of eight rows at most."""
    capacity = 64 * 32
    for live in (1, 2, 8, 9, 33, 64):
        share = [0] * DIES
        for die, first, rows, part in dealing(capacity, I, F32, Q_REUSE_MOE, True):
            share[die] += sum(1 for row in range(first, first + rows) if row < live * 32 and part == 0)
        assert sum(share) == live * 32 and max(share) - min(share) <= 8, (live, share)


def test_unaligned_fp32_rows_go_round_robin(dealing):
    """fp32 rows that are fetched element by element: one row per workgroup, round-robin over the dies, while a
    compute unit gets at most two of up to 8192 elements; four rows per workgroup beyond.  Aligned rows, fp16 rows
    and longer rows keep their ranges."""
    for M, K in ((16, 2050), (61, 2050), (250, 8191), (512, 4099), (300, 8190)):
        assert dealing(M, K, F32, Q_W8_DYNAMIC) == [(m % DIES, m, 1, 0) for m in range(M)], (M, K)
    for M, K in ((513, 2050), (560, 4099), (700, 8191)):
        assert all(rows == 4 for _, _, rows, _ in dealing(M, K, F32, Q_W4A8)), (M, K)
    for M, K, dtype in ((61, 2048, F32), (61, 2050, F16), (250, 9001, F32), (560, 4099, F16)):
        got = dealing(M, K, dtype, Q_W8_DYNAMIC)
        for die in range(DIES):
            mine = [first for d, first, rows, _ in got if d == die]
            assert mine == list(range(mine[0], mine[0] + len(mine))), (M, K, dtype)
