// Few rows (2 .. 64, few_cols says where): gemm_few_kernel, one workgroup of eight waves per 16 or 32
// columns, K interleaved over the waves, operands straight to registers.  Bound by HBM.
#include "rk_kernels_common.h"

namespace {

constexpr int FEW_WAVES = 8;

// CW = 16: v_mfma_i32_16x16x64_i8, RG groups of 16 rows; a load instruction covers the workgroup's 16
// columns of two consecutive k-tiles (int4: super-tiles).  CW = 32: v_mfma_i32_32x32x32_i8, RG blocks of
// 32 rows.  Either way a step of a wave is one 1 KiB load of weights, which is the first MFMA operand as a
// lane holds it, and one (int4: two) of activations per row group, the second one.
//
// What bounds it: bytes in flight.  The streaming kernel's 32-column tiles gave 16 rows of 14336 x 4096
// 128 workgroups of four waves with 3 KiB of weights each on their way -- 1.5 MB for the whole chip, where
// 7 TB/s at a microsecond's latency need 7 -- and took 20.4 us for 58.7 MB.  16 columns give every compute unit a
// workgroup, eight waves ask for eight KiB each (16 MB in all): 11.6 us.  A workgroup pulls as many activation bytes
// as weights through its compute unit (from L2; rows past M are not fetched), which is why more rows want
// 32 columns, and many rows the other kernels.  Loads go through bounds-checked descriptors: steps past the
// end of K return zeros without touching memory, so no branch stands around a load and the compiler
// counts the outstanding ones exactly.
template <int EPI, bool W4, int CW, int RG>
__global__ __launch_bounds__(FEW_WAVES * 64) void gemm_few_kernel(const uint8_t* h_A, const uint8_t* h_W, int h_M, int h_K,
                                                                  rkh_gemm_args g) {
    g.A = h_A; g.W = h_W; g.M = h_M; g.K = h_K;
    constexpr int AT = W4 ? 2 : 1, TPL = 32 / CW;
    constexpr int CREGS = CW == 32 ? 16 : 4, QUADS = RG * CREGS / 4;
    constexpr int LPS = 1 + AT * RG;                       // loads of a step
    constexpr int R = LPS <= 2 ? 8 : LPS == 3 ? 6 : 4;     // steps in flight
    using acc_t = typename std::conditional<CW == 32, v16i, v4i>::type;
    __shared__ __attribute__((aligned(16))) v4i red[FEW_WAVES][QUADS][64];
    const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane(wave_id());
    const int half = (lane / CW) & 1, sub = lane / (2 * CW);
    const int KB = (int)rkh_align_up(g.K, RKH_K_ALIGN) / 32;
    const int p = (int)blockIdx.x / TPL, col0 = (int)blockIdx.x % TPL * CW;
    const int steps = KB / (AT * TPL);
    const int mine = steps > wave ? (steps - wave + FEW_WAVES - 1) / FEW_WAVES : 0;

    const size_t block_bytes = (size_t)(KB / AT) * 1024; // one column block (int4: of super-tiles) over all of K
    const __amdgpu_buffer_rsrc_t wrsrc =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(g.W) + (size_t)p * block_bytes, 0, (int)block_bytes, 0x00020000);
    const unsigned w_lane = (unsigned)sub * 1024u + (unsigned)(col0 + lane % CW + 32 * half) * 16u;
    __amdgpu_buffer_rsrc_t arsrc[RG];
    unsigned a_lane[RG];
#pragma unroll
    for (int i = 0; i < RG; ++i) {
        const int row = i * CW + lane % CW; // (16-row groups pair up in a 32-row block of the tiled rows)
        arsrc[i] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(g.A) + (size_t)(i * CW / 32) * KB * 1024, 0, KB * 1024, 0x00020000);
        a_lane[i] = row < g.M ? (unsigned)(sub * AT) * 1024u + (unsigned)(row % 32 + 32 * half) * 16u : 0xFFFFFFF0u;
    }

    // the scales of the outputs this wave will finish, ahead of everything
    float as = 0.0f, ws[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    const int rg = wave / (CREGS / 4), quad = wave % (CREGS / 4); // of the quad of sums this wave finishes (wave < QUADS)
    const int m = rg * CW + lane % CW;
    const int n0 = block_first_col(p, g.interleave_F) + col0 + 8 * quad + 4 * (lane / CW);
    const bool block_live = g.interleave_F ? p < g.N / 32 : true;
    if constexpr (EPI != RKH_EPI_I32) {
        if (wave < QUADS) {
            as = g.a_scale[m < g.M ? m : 0];
#pragma unroll
            for (int r = 0; r < 4; ++r) ws[r] = g.w_scale[n0 + r < g.N ? n0 + r : 0];
        }
    }

    acc_t acc[RG];
#pragma unroll
    for (int i = 0; i < RG; ++i)
#pragma unroll
        for (int r = 0; r < CREGS; ++r) acc[i][r] = 0;
    v4i w[R], a[R][RG * AT];
    auto issue = [&](int slot, int step) {
        const bool in = step < steps;
        const unsigned at = (unsigned)step * (unsigned)(TPL * 1024);
        w[slot] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wrsrc, (int)(in ? at + w_lane : 0xFFFFFFF0u), 0, 2 /* streaming */));
#pragma unroll
        for (int i = 0; i < RG; ++i)
#pragma unroll
            for (int t = 0; t < AT; ++t)
                a[slot][i * AT + t] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(
                    arsrc[i], (int)(in && a_lane[i] != 0xFFFFFFF0u ? at * AT + a_lane[i] + t * 1024u : 0xFFFFFFF0u), 0, 0));
    };
    auto multiply = [&](int slot) {
#pragma unroll
        for (int t = 0; t < AT; ++t) {
            v4i op = w[slot];
            if constexpr (W4) { // 16 x code: the two words of this half of the super-tile
                const int x = t ? w[slot].z : w[slot].x, y = t ? w[slot].w : w[slot].y;
                op = v4i{(x << 4) & (int)0xF0F0F0F0, x & (int)0xF0F0F0F0, (y << 4) & (int)0xF0F0F0F0, y & (int)0xF0F0F0F0};
            }
#pragma unroll
            for (int i = 0; i < RG; ++i) {
                if constexpr (CW == 32) acc[i] = __builtin_amdgcn_mfma_i32_32x32x32_i8(op, a[slot][i * AT + t], acc[i], 0, 0, 0);
                else acc[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(op, a[slot][i * AT + t], acc[i], 0, 0, 0);
            }
        }
    };
#pragma unroll
    for (int r = 0; r < R; ++r) issue(r, wave + r * FEW_WAVES);
    int next = wave + R * FEW_WAVES, left = mine;
    for (; left > R; left -= R) {
#pragma unroll
        for (int r = 0; r < R; ++r) {
            multiply(r);
            issue(r, next);
            next += FEW_WAVES;
        }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) multiply(r); // (steps past the end of K: weights of zero)

#pragma unroll
    for (int i = 0; i < RG; ++i)
#pragma unroll
        for (int q = 0; q < CREGS / 4; ++q)
            red[wave][i * (CREGS / 4) + q][lane] = v4i{acc[i][q * 4], acc[i][q * 4 + 1], acc[i][q * 4 + 2], acc[i][q * 4 + 3]};
    __syncthreads();
    if (wave >= QUADS) return;
    v4i sum = red[0][wave][lane];
#pragma unroll
    for (int v = 1; v < FEW_WAVES; ++v) sum += red[v][wave][lane];
    if (m >= g.M || !block_live) return;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (n0 + r < g.N) store_out(g.C, EPI, (size_t)m * g.ldc + n0 + r, W4 ? sum[r] >> 4 : sum[r], as, ws[r]);
    }
}

template <int CW, int RG>
int launch_few(hipStream_t st, const rkh_gemm_args& g) {
    const dim3 grid((g.N + CW - 1) / CW), block(FEW_WAVES * 64);
    // (int4 weights: 16 columns only, see few_cols)
#define RK_FEW(EPI)                                                                                                         \
    do {                                                                                                                    \
        if (!g.w_int4) hipLaunchKernelGGL((gemm_few_kernel<EPI, false, CW, RG>), grid, block, 0, st, g.A, g.W, g.M, g.K, g); \
        else if constexpr (CW == 16)                                                                                        \
            hipLaunchKernelGGL((gemm_few_kernel<EPI, true, CW, RG>), grid, block, 0, st, g.A, g.W, g.M, g.K, g);            \
        else return RKH_ERR_RUNTIME;                                                                                        \
    } while (0)
    mark(st, "gemm_few_kernel");
    switch (g.epilogue) {
    case RKH_EPI_I32: RK_FEW(RKH_EPI_I32); break;
    case RKH_EPI_F16: RK_FEW(RKH_EPI_F16); break;
    case RKH_EPI_F32: RK_FEW(RKH_EPI_F32); break;
    default: return RKH_ERR_RUNTIME;
    }
#undef RK_FEW
    RKH_CHECK(hipGetLastError());
    return RKH_OK;
}

} // namespace

namespace rkk {
// Columns of a workgroup, or 0 where another kernel is better.  Both sides measured with fp16 rows,
// quantization included, weights from HBM, us.
int few_cols(const rkh_gemm_args& g) {
    if (g.blk_expert || g.epilogue == RKH_EPI_SWIGLU || g.M < 2 || g.M > 64) return 0;
    // (tuning aids that say how one of the kernels below is used, or up to which row: the calls they mean are theirs)
    static const bool decode_forced = getenv("RK_NPU_HIP_GEMV_COLS") || getenv("RK_NPU_HIP_GEMV_MAX_ROWS");
    static const bool stream_forced = getenv("RK_NPU_HIP_STREAM_MAX_ROWS") != nullptr;
    if (stream_forced || (decode_forced && g.M <= 8)) return 0;
    // int4 weights ride as 16 * code: the int32 sum of more than 2^17 k may wrap.  int8: the kernel's descriptors
    // hold the bytes of a column block over all of K, 32 K, in 32 bits, and K = 2^27 would read as none; the
    // line lies well before that, and beyond anything measured here.
    if (g.K > (g.w_int4 ? 1 << 17 : 1 << 24)) return 0;
    const long kp = (long)rkh_align_up(g.K, RKH_K_ALIGN);
    const bool narrow = g.N <= 4096; // at most one workgroup of 16 columns per compute unit
    if (g.M <= 8) {
        // The decode kernel keeps the rows that its staging area holds at once (and quantizes them itself);
        // beyond, it walks K in chunks behind a quantization launch.  int4, five to eight rows: 6144 x 4096
        // 10.2 -> 8.5, 11008 x 4096 13.1 -> 11.1, 14336 x 4096 15.6 -> 13.2; three / four 14.8 -> 13.1, 11008 x 2048
        // 11.8 -> 10.2; two of 20000 x 2048 18.6 -> 17.2.  Wider int4 matrices stay (8192 x 8192 12.1 against 13.2).
        // int8: 14336 x 4096 21.4 -> 16.4, 11008 x 4096 18.0 -> 13.9, 11008 x 11008 32.5 -> 26.0, 28672 x 8192 two rows
        // 51.1 -> 48.9 -- and from five rows of K = 8192 on, although they would fit: 8192 x 4096 five / eight rows
        // 11.5 / 14.6 -> 10.9 / 11.1, 8192 x 8192 16.8 / 19.7 -> 15.9 / 15.8 (6144 x 4096 six rows a tie).
        const long rows = g.M == 2 ? 2 : g.M <= 4 ? 4 : 8;
        const bool staged = kp * rows <= (rows >= 4 && !g.w_int4 ? 65536 : 32768);
        if (g.w_int4) return !staged && narrow ? 16 : 0;
        // (8192 x 13312 five / six / seven rows 22.1 / 23.1 / 24.0 -> 23.4 / 23.5 / 23.5, 14336 23.2 / 24.5 / 25.3 -> 23.9; 12288 and
        // 16384 columns are ahead from five rows on.)
        if (staged && g.M <= 6 && g.N > 12288 && g.N < 16384) return 0;
        return !staged || (g.M > 4 && kp >= 8192) ? 16 : 0;
    }
    if (g.w_int4) {
        // 4096 x 2048 16 / 32 rows 9.2 / 10.2 -> 7.8 / 8.9, 4096 x 4096 9.1 / 9.4 -> 7.9 / 9.2, 14336 x 4096 15.7 -> 14.0 at 16 rows
        // but 16.6 against 18.2 at 32; wider matrices lose (4096 x 5120 a tie, 4096 x 11008 11.2 against 13.2).
        return narrow && (g.M <= 16 || (g.M <= 32 && kp <= 8192)) ? 16 : 0;
    }
    // int8, 16 rows: 4096 x 4096 11.8 -> 8.7, 11008 x 4096 21.5 -> 14.4, 14336 x 4096 26.0 -> 17.1, 28672 x 4096 48.2 -> 32.4;
    // 32 columns 4096 x 8192 12.3 -> 11.0, 4096 x 11008 15.5 -> 14.7, 4096 x 28672 27.7 -> 24.8, 13824 x 5120 26.2 -> 21.0.
    // What lies just past the 2048 k that the eight waves' first eight loads cover waits for memory once more:
    // 2304 x 4128 16 / 32 rows 8.25 / 8.75 -> 8.95 / 9.7 (2048 9.0 -> 7.4 at 5120, 2304 x 8192 10.2 -> 9.5).
    if (kp == 2304 && g.N > 4096 && g.N <= 6144) return 0;
    if (g.M <= 16 && g.N > 8192) { // more than a workgroup per compute unit
        // The same, 16 rows: 2304 x 9216 / 14336 / 28672 11.8 / 12.4 / 19.6 -> 12.6 / 12.9 / 20.1, 2560 x 9216 12.1 -> 12.7 (20480 18.7 -> 16.8,
        // 2816 x 9216 12.85 -> 12.7); past two rounds 4608 x 9216 16.6 -> 17.0 (12288 a tie).  Short K: 512 x 20480 9.45 -> 10.4, 1024 x
        // 28672 12.5 -> 13.5 (1024 x 20480 12.0 -> 11.4).  K = 8192 is slow here (8192 x 8320 24.4 where 7936 takes 21.6 and 8448 24.4;
        // not for the channels that its power-of-two blocks share: starting each block at another k made it 26.3):
        // 8320 / 10240 / 13312 / 28672 columns 23.8 / 24.8 / 26.25 / 47.4 -> 24.5 / 25.5 / 26.75 / 48.8 (8192 19.4 -> 18.6, 20480 42.8 ->
        // 37.8, 30720 50.9 -> 49.7).
        if (kp > 2048 && kp < 2816 && (g.N <= 16384 || g.N > 24576)) return 0;
        if (kp > 4096 && kp < 4864 && g.N < 12288) return 0;
        if (kp < 2048 && g.N > (kp < 1024 ? 16384 : 24576)) return 0;
        if (kp == 8192 && (g.N < 14336 || (g.N > 24576 && g.N < 29696))) return 0;
    }
    if (g.M <= 16) return narrow ? 16 : g.N <= 32768 ? 32 : 0;
    // 32 rows: 4096 x 4096 11.8 -> 10.3, 11008 x 4096 22.4 -> 18.1, 28672 x 4096 50.0 -> 42.0; 32 columns 4096 x 8192 12.9 -> 12.0,
    // 13824 x 5120 27.4 -> 25.4; 4096 x 12288 16.2 against 17.6: an activation tile for every weight tile is too much there.
    if (g.M <= 32) return narrow ? 16 : g.N <= 8192 ? 32 : 0;
    // 33 to 64 rows, 32 columns.  Up to 4096 columns the streaming kernel has tiles of 32 columns: 11008 x 4096 22.2 against 24.
    if (narrow) return 0;
    if (g.N <= 8192) {
        // 40 / 64 rows: 4096 x 5120 14.6 / 14.7 -> 12.9 / 14.6, 4096 x 8192 15.7 / 16.4 -> 13.4 / 15.7, 13824 x 5120 33.6 / 34.0 ->
        // 28.1 / 32.5, 2560 x 4128 10.65 / 10.7 -> 10.4 / 10.75, 1024 x 4128 8.6 / 8.55 -> 7.9 / 8.3.  In between, 40 / 48 / 64 rows:
        // 2048 x 4128 8.7 / 8.7 / 8.8 -> 9.5 / 9.8 / 10.4, 2048 x 5120 9.8 / 9.9 / 9.9 -> 9.6 / 9.9 / 10.9, 1536 x 5120 8.35 / 8.35 /
        // 8.4 -> 8.3 / 8.5 / 9.05, 2048 x 7168 10.5 / 10.6 / 10.7 -> 10.3 / 10.4 / 11.05, 2048 x 8192 10.8 / 10.8 / 10.95 -> 9.9 / 10.2 / 10.6.
        const int most = kp <= 1024 || kp >= 2560 || g.N > 7680 ? 64 : g.N > 6144 ? 48 : g.N >= 5120 ? 40 : 0;
        return g.M <= most ? 32 : 0;
    }
    // Wider, more than a workgroup per compute unit.  Up to 8448 columns, 264 tiles of the streaming kernel, that one is
    // ahead (3072 x 8320 40 / 56 rows 15.0 / 15.15 -> 14.7 / 16.0, 5120 x 8448 21.65 / 22.0 -> 21.9 / 23.6, 8192 x 8320 29.2 / 30.1 ->
    // 33.3 / 36.0); with 266 tiles it takes 15 % longer (3072 x 8512 17.2).  Beyond, 40 / 56 rows: 3072 x 8512 17.2 / 17.5 -> 14.9 / 16.3,
    // 4096 x 12288 21.9 / 22.5 -> 19.6 / 21.7 (64: 22.5 -> 23.4), 14336 x 14336 61.3 / 62.3 -> 50.2 / 57.4; K = 8192 48 / 56 rows
    // 8704 columns 35.1 / 35.7 -> 35.0 / 36.3, 12288 36.7 / 37.2 -> 36.2 / 37.9; 2048 x 9216 40 / 48 / 56 rows 14.1 / 14.2 / 14.2 ->
    // 13.7 / 14.2 / 14.6; 1024 x 9216 9.9 -> 10.5 at 40.
    if (g.N <= 8448 || g.N > 14336) return 0;
    const int most = kp == 8192 ? 48 : kp >= 3072 ? 56 : kp >= 2048 ? 40 : 0;
    return g.M <= most ? 32 : 0;
}
int launch_gemm_few(hipStream_t st, const rkh_gemm_args& g, int cols) {
    if (cols == 16) return g.M <= 16 ? launch_few<16, 1>(st, g) : launch_few<16, 2>(st, g);
    return g.M <= 32 ? launch_few<32, 1>(st, g) : launch_few<32, 2>(st, g);
}
} // namespace rkk
