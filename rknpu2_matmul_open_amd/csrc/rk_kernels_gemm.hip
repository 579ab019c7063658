// int8 MFMA GEMM for prefill-sized M: gemm_wk_kernel (tiles of 32..128 rows x 256 columns,
// activations through an LDS ring, waves split K), gemm_wk_reduce_kernel (sum of K-split
// partial tiles + epilogue) and their launcher.  Bound by the matrix pipes.
#include "rk_kernels_tile.h"

namespace {

// ---- tiles of (32 * TM) rows x (128 * TN) columns ------------------------------
// v_mfma_i32_16x16x64_i8.  Large launches run at the clock that the power limit leaves, so energy per product
// is what counts: a loop of nothing but MFMAs on quantized activations (codes of N(0, 2.5) with outliers) and
// N(0, 30) weights reaches 3.53 POP/s with 32x32x32 and 4.19 with 16x16x64 (int4 weights as 16 * code: 3.77 and 4.67).
// Calls with quantization, us, from the kernel of 32x32x32 products whose sub-steps issued their loads together to this one, one
// box, two sets of operands in turn (partly from the last-level cache): int4 2048 x 4096 x 4096 38.3 -> 33.2, 4096^3 67.1 -> 59.4, 512 x
// 14336 x 4096 36.9 -> 33.4, int8 4096 x 4096 x 14336 205 -> 188, 1000 x 4096 x 4096 26.3 -> 23.0, the FFN 4096 -> 14336 -> 4096 of
// 128 / 512 rows 42.7 -> 39.6 / 101 -> 94 (weights from memory: 48.7 -> 47.3 / 105 -> 98).  Of 260 shapes drawn from 65 - 4096
// rows, 512 - 14336 columns and k one that this kernel serves is slower beyond the noise of three runs: int8 1241 x 13825 x 1152 71.1 -> 71.25.
//
// Eight waves = 4 column groups (wn) x 2.  In the tiles of up to 128 rows the two waves of a column group
// split K (k-half wk): each accumulates all rows x 32 * TN columns over every second 128 k, and the halves are
// summed once, through LDS, before the epilogue -- no weight byte is loaded (or unpacked) by two waves.  In
// the tiles of 256 x 256 (RS) they split the rows (row half wk): 128 x 64 each over the whole K, no exchange.
//
// For a wave K goes in units of 64 k: RM activation operands of 16 rows and CN weight operands of 16 columns, RM x CN MFMAs.
// A step -- what is copied to LDS at a time -- is one or two units of every wave (two where int4 super-tiles are
// shared by a pair of units, and where one would be less than 8 KiB of activations).  A k-tile is 32 rows x 32 k with 16 bytes per lane; operand lane (r, q) = (l % 16, l / 16)
// takes row 16 h + r, k-half q % 2 of k-tile q / 2 of the unit's two, i.e. both operands are read with per-lane addresses in
// pieces of 256 contiguous bytes (which k a lane group holds is free as long as both operands agree).  Int4 super-tiles
// hold 64 k in 16 bytes per lane: one load brings the words of both units, lane group q the k-half q % 2 of super-tile
// q / 2 of the step's two, and unit u takes k-tile u of each.
//
// Activations: every wave copies NC KiB of a step global -> LDS directly (no registers), D steps ahead, into a
// ring of NBUF buffers.  Weights: global -> registers, NSW - 1 units ahead (int4: steps).  An operand of the next
// unit is read from LDS into the registers of the one that the last CN MFMAs have used, and waited for one unit later:
// LDS reads complete in order, so a counted wait leaves the younger RM - 1 in flight.
//
// The loads of a unit are spread between its MFMAs.  Issued together behind a barrier, the eight waves' loads queue in front of
// the compute unit's 64 B per clock and a wave stands still until its own have been taken (256 x 256 tiles, int8:
// 1274 cycles per 64 k of which 1024 are MFMAs; spread 1124).
//
// All loads of the loop are inline assembly and every wait is explicit.  (The compiler's own bookkeeping orders each
// LDS read after ALL outstanding global -> LDS copies, which would undo the prefetch.)  The waits rely on vector
// memory loads completing in issue order and on every unit issuing the same loads -- copies first, then weights -- also
// beyond the end of K, where the source pointers stop advancing (those loads hit the L1 and nothing uses them):
//  * weights: unit t ends with the wait for those of unit t + 1, issued in unit t + 2 - NSW; the loads of the
//    NSW - 2 units since may be outstanding.  (int4: the second unit of step s waits, ahead of its unpacking, for the
//    weights of step s + 1, issued in the first unit of step s + 2 - NSW.)
//  * publication: between the barrier at the end of step B and the next one, G steps later, waves read operands of steps up to
//    B + G + 1.  Those were copied in steps up to B + G + 1 - D: the last wait ahead of the barrier leaves no older copy
//    in flight (in_flight() is the smaller of the two bounds).
//  * reuse: the copy issued in step s overwrites the buffer of step x = s + D - NBUF, whose last reads were
//    issued in the first unit of step x and waited for in its second, ahead of the barrier that ends a step in x .. s - 1
//    (needs NBUF >= D + G).
//
// Split K over workgroups (ksplit > 1, small M): every part stores its int32
// tile in accumulator order to scratch and gemm_wk_reduce_kernel, launched
// behind it, adds the parts and runs the epilogue.  (Summing inside this
// kernel, in the part that arrives last, needs a device-scope release per
// workgroup; on this multi-die part each one walks the die's L2, and 32
// workgroups per die queueing for that cost more than the second launch.)
constexpr int WK_RING_BYTES = 128 * 1024;
constexpr int WK_SCALES_OFF = WK_RING_BYTES;                      // fp32 scales of the tile: 256 rows, then 256 columns; twice
constexpr int WK_ROW_SCALES = 256, WK_SCALES = (WK_ROW_SCALES + 256) * 4;
constexpr int WK_STAGE_OFF = WK_SCALES_OFF + 2 * WK_SCALES, WK_STAGE = 16 * 144; // per wave: 16 rows x 32 columns
constexpr int WK_LDS_BYTES = WK_STAGE_OFF + 8 * WK_STAGE;
constexpr int WK_PART_K = 256;                                    // granularity of a K split over workgroups

typedef __attribute__((address_space(3))) uint8_t* lds_ptr_t;

// Row / column block of logical dense tile `tile`: column sweeps over groups of
// 4 row blocks, so that concurrently running tiles share weight columns in L2.
// (unsigned arithmetic: these divisions stand between a wave's start and its first load, and a
// signed division by a run-time value is half as long again)
__device__ __forceinline__ void wk_tile_coords(unsigned tile, unsigned mblocks, unsigned nblocks, int& mblk, int& nblk) {
    constexpr unsigned GM = 4;
    const unsigned per_group = GM * nblocks;
    const unsigned group = tile / per_group;
    const unsigned first_m = group * GM;
    const unsigned gm = min(mblocks - first_m, GM);
    const unsigned in_group = tile - group * per_group;
    const unsigned col = in_group / gm;
    mblk = (int)(first_m + in_group - col * gm);
    nblk = (int)col;
}

// ---- 16 x 16 accumulator tiles --------------------------------------------------
// The weights are the FIRST MFMA operand: lane (r, q) owns output row r of the tile and its columns 4 q .. 4 q + 3.
// Two neighbouring tiles make a unit of 16 rows x 32 columns, the width of a column block.

// Stage a unit in the wave's staging area and read it back as 16-byte pieces of rows.  LDS operations of a wave complete in
// issue order, so nothing is waited for between the two, or ahead of the next unit; the fence keeps the compiler from swapping them.
template <typename T>
struct StagedUnit {
    static constexpr int ES = sizeof(T), PITCH = 32 * ES + 16, PIECES = ES / 2; // 16-byte pieces of a lane
    v4i piece[PIECES];
    __device__ __forceinline__ void exchange(const T (&vals)[8], uint8_t* stage, int lane) {
        const int r = lane & 15, q = lane >> 4;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            T* dst = reinterpret_cast<T*>(stage + r * PITCH + (16 * h + 4 * q) * ES);
#pragma unroll
            for (int e = 0; e < 4; ++e) dst[e] = vals[4 * h + e];
        }
        asm volatile("" ::: "memory");
#pragma unroll
        for (int t = 0; t < PIECES; ++t) {
            const int c = lane + 64 * t;
            piece[t] = *reinterpret_cast<const v4i*>(stage + c / (2 * ES) * PITCH + c % (2 * ES) * 16);
        }
    }
    template <bool ALL_ROWS>
    __device__ __forceinline__ void store(T* C, int ldc, int m0, int n0, int m_limit, int lane) const {
#pragma unroll
        for (int t = 0; t < PIECES; ++t) {
            const int c = lane + 64 * t, row = c / (2 * ES);
            if (ALL_ROWS || m0 + row < m_limit) // the output is not read again by this kernel: streaming store
                __builtin_nontemporal_store(piece[t], reinterpret_cast<v4i*>(reinterpret_cast<uint8_t*>(C) + ((size_t)(m0 + row) * ldc + n0) * ES +
                                                                             c % (2 * ES) * 16));
        }
    }
};

// A unit whose columns end inside it, or whose rows are not 16-byte aligned in C.
template <typename T>
__device__ __forceinline__ void store_unit_plain(T* C, int ldc, int m0, int n0, int m_limit, int n_limit, const T (&vals)[8], int lane) {
    const int m = m0 + (lane & 15);
    if (m >= m_limit) return;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int n = n0 + 16 * (e >> 2) + 4 * (lane >> 4) + (e & 3);
        if (n < n_limit) C[(size_t)m * ldc + n] = vals[e];
    }
}

template <int EPI>
using wk_out_t = typename std::conditional<EPI == RKH_EPI_I32, int, typename std::conditional<EPI == RKH_EPI_F16, __half, float>::type>::type;

// Scale, convert and store ROWS x (16 * CN) sums of a wave: acc_of(i, j) is the tile of rows m0 + 16 i and physical columns
// pb0 * 32 + 16 j, as(i) / ws(j, e) the lane's row scale and column scales.
template <int ROWS, int CN, bool W4, int EPI, class Acc, class RowScale, class ColScale>
__device__ __forceinline__ void wk_store(const rkh_gemm_args& g, Acc&& acc_of, RowScale&& as, ColScale&& ws, int m0, int pb0,
                                         int m_limit, uint8_t* stage, int lane) {
    using T = wk_out_t<EPI>;
    constexpr bool SWIGLU = EPI == RKH_EPI_SWIGLU;
    constexpr int NB = SWIGLU ? 1 : CN / 2; // column blocks stored per 16 rows
    T* C = static_cast<T*>(g.C);
    int n0[NB], n_end = SWIGLU ? g.interleave_F : g.N;
    bool live[NB], whole[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        // padding blocks beyond the matrix hold zeros; with interleaved columns their logical index would alias a real
        // column, so the block itself is tested
        const int pb = pb0 + b;
        n0[b] = SWIGLU ? (pb0 >> 1) * 32 : block_first_col(pb, g.interleave_F);
        live[b] = SWIGLU ? n0[b] < n_end : g.interleave_F ? pb < g.N / 32 : pb * 32 < g.N;
        whole[b] = n0[b] + 32 <= n_end &&
                   ((reinterpret_cast<uintptr_t>(C) | ((size_t)g.ldc * sizeof(T)) | ((size_t)n0[b] * sizeof(T))) & 15) == 0;
    }
    uint32_t bits[ROWS];
    const auto values = [&](T (&vals)[8], int i, int b) {
        uint32_t top = 0;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int j = 2 * b + (e >> 2);
            int sum = acc_of(i, j)[e & 3];
            if (W4) sum >>= 4;
            if constexpr (EPI == RKH_EPI_I32) {
                vals[e] = sum;
            } else if constexpr (SWIGLU) {
                int up = acc_of(i, CN / 2 + j)[e & 3];
                if (W4) up >>= 4;
                const float gate = dequant(sum, as(i), ws(j, e & 3));
                const float y = __fmul_rn(silu_poly(gate), dequant(up, as(i), ws(CN / 2 + j, e & 3)));
                top = max(top, __float_as_uint(y) & 0x7fffffffu);
                vals[e] = y;
            } else if constexpr (EPI == RKH_EPI_F16) {
                vals[e] = __float2half_rn(dequant(sum, as(i), ws(j, e & 3)));
            } else {
                vals[e] = dequant(sum, as(i), ws(j, e & 3));
            }
        }
        bits[i] = top;
    };
    bool full = m0 + 16 * ROWS <= m_limit;
#pragma unroll
    for (int b = 0; b < NB; ++b) full = full && live[b] && whole[b];
    if (full) { // straight-line code: a unit is stored behind the exchange of the next one
        StagedUnit<T> held[2];
#pragma unroll
        for (int u = 0; u < ROWS * NB; ++u) {
            T vals[8];
            values(vals, u / NB, u % NB);
            held[u & 1].exchange(vals, stage, lane);
            if (u > 0) held[(u - 1) & 1].template store<true>(C, g.ldc, m0 + 16 * ((u - 1) / NB), n0[(u - 1) % NB], m_limit, lane);
        }
        held[(ROWS * NB - 1) & 1].template store<true>(C, g.ldc, m0 + 16 * (ROWS - 1), n0[NB - 1], m_limit, lane);
    } else {
#pragma unroll
        for (int u = 0; u < ROWS * NB; ++u) {
            const int i = u / NB, b = u % NB;
            if (!live[b]) continue;
            T vals[8];
            values(vals, i, b);
            StagedUnit<T> unit;
            if (whole[b]) {
                unit.exchange(vals, stage, lane);
                unit.template store<false>(C, g.ldc, m0 + 16 * i, n0[b], m_limit, lane);
            } else {
                store_unit_plain(C, g.ldc, m0 + 16 * i, n0[b], m_limit, n_end, vals, lane);
            }
        }
    }
    if constexpr (SWIGLU) {
        if (g.row_max_bits && live[0]) { // largest |middle| per row and 32 columns
#pragma unroll
            for (int i = 0; i < ROWS; ++i) {
                uint32_t top = max(bits[i], (uint32_t)__shfl_xor((int)bits[i], 16));
                top = max(top, (uint32_t)__shfl_xor((int)top, 32));
                const int m = m0 + 16 * i + lane;
                if (lane < 16 && m < m_limit) g.row_max_bits[(size_t)m * (n_end / 32) + (pb0 >> 1)] = top;
            }
        }
    }
}

// NAMED: x becomes valid -- what keeps the compiler's own products behind the wait; for products that are asm statements their
// order is enough, and a statement that "writes" an operand would get a wait state behind it.
template <int N, bool NAMED> __device__ __forceinline__ void wait_lds(v4i& x) {
    if constexpr (NAMED) asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(x) : "n"(N) : "memory");
    else asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory");
}
template <int OFF> __device__ __forceinline__ void read_lds(v4i& x, uint32_t addr) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(x) : "v"(addr), "n"(OFF));
}
template <int OFF> __device__ __forceinline__ void load_regs(v4i& x, unsigned lane_off, const uint8_t* base) {
    asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3" : "=v"(x) : "v"(lane_off), "s"(base), "n"(OFF));
}
__device__ __forceinline__ void load_far(v4i& x, const uint8_t* src) { asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(x) : "v"(src)); }
// The product as an asm statement, for the chained tiles: sums stay in one place (of products that it knows the compiler rotated 128
// sums through the register file, and with the next tile's weights beside them spilled some around the tile's first products).
// What the compiler then does not order: a vector instruction that writes an operand has to be two wait states ahead
// of the product -- the weights are unpacked well ahead --, and one that reads a sum waits for the last products, settle().
// The build checks both in the compiled code (audit_waits.py).
__device__ __forceinline__ void mfma(v4i& sum, const v4i& w, const v4i& a) {
    asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, %0" : "+v"(sum) : "v"(w), "v"(a));
}
__device__ __forceinline__ void mfma_first(v4i& sum, const v4i& w, const v4i& a) {
    asm volatile("v_mfma_i32_16x16x64_i8 %0, %1, %2, 0" : "=&v"(sum) : "v"(w), "v"(a));
}
__device__ __forceinline__ void keep(v4i& x) { asm volatile("" : "+v"(x)); }

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm" // m0 is set and clobbered on purpose below
// 16 bytes per lane, lane-contiguous, global -> LDS; the offset counts on both sides.  A load to LDS needs a wait state
// behind a scalar write of M0, which the compiler does not insert into an asm statement (the build checks for it): the
// change of the wave's priority is put there.
template <int OFF, int PRIO> __device__ __forceinline__ void copy_lds(unsigned lane_off, const uint8_t* src, uint32_t dst) {
    asm volatile("s_mov_b32 m0, %2\n\ts_setprio %4\n\tglobal_load_lds_dwordx4 %0, %1 offset:%3" ::"v"(lane_off), "s"(src), "s"(dst), "n"(OFF), "n"(PRIO)
                 : "memory", "m0");
}
// The same for the lanes of a mask (every lane is active here, and is again behind the copy).
template <int OFF, int PRIO> __device__ __forceinline__ void copy_lds(unsigned lane_off, const uint8_t* src, uint32_t dst, unsigned long long lanes) {
    asm volatile("s_mov_b32 m0, %2\n\ts_setprio %4\n\ts_mov_b64 exec, %5\n\tglobal_load_lds_dwordx4 %0, %1 offset:%3\n\ts_mov_b64 exec, -1" ::"v"(lane_off),
                 "s"(src), "s"(dst), "n"(OFF), "n"(PRIO), "s"(lanes) : "memory", "m0");
}
__device__ __forceinline__ void copy_lds_dword(const float* src, uint32_t dst) { // 4 bytes per lane, likewise
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dword %0, off" ::"v"(src), "s"(dst) : "memory", "m0");
}
#pragma clang diagnostic pop

// The shape of a tile and of its pipeline.
template <int TM, bool W4, int TN, bool RS>
struct WkShape {
    static_assert(!RS || (TM == 4 && TN == 2), "row-split waves: tiles of 256 x 256");
    static constexpr bool ONE = TM == 4 && !W4;                 // a step is one unit
    static constexpr bool ASM = RS;                             // products as asm statements, see mfma()
    static constexpr int U = ONE ? 1 : 2;
    static constexpr int RM = 2 * TM, CN = 2 * TN;              // operands of 16 rows / columns per wave
    static constexpr int BM = RS ? 256 : 32 * TM;               // rows of a tile
    static constexpr int KT = (RS ? 2 : 4) * U;                 // k-tiles of a step
    static constexpr int BUF = BM / 32 * KT * 1024, NBUF = ONE ? (RS ? 8 : 6) : TM == 4 ? 4 : 8;
    static constexpr int NC = BUF / 8192;                       // 1 KiB copies of a wave per step
    static constexpr int NW = CN;                               // weight loads per unit (int4: per step, in its first unit)
    static constexpr int NSW = ONE ? (RS ? 4 : 3) : TM == 4 ? 2 : 4; // slots of the weight ring
    static constexpr int G = ONE || (W4 && TM < 4) ? 2 : 1;             // steps between barriers
    static constexpr int D = ONE ? 4 : W4 && TM < 4 ? 5 : 3;         // look-ahead of the copies
    static constexpr int UNR = RS ? NBUF / 2 : NBUF;            // steps of an unrolled trip (RS: 256 k, half the ring)
    // RS: the step of a trip whose copies (weights) are a tile's last ones: in the tile's last trip but one (last trip)
    static constexpr int A_TURN = ((-D - 1) % UNR + UNR) % UNR, W_TURN = (-(W4 ? NSW - 1 : (NSW - 1) / U) - 1 + 2 * UNR) % UNR;
    static_assert(!RS || ((D + UNR - 1) / UNR == (A_TURN == UNR - 1 ? 1 : 2) && W_TURN == 0 && NSW - 1 < UNR * (W4 ? 1 : U)), "the trips of the turns");
    static constexpr int copies(int unit) { return U == 1 ? NC : NC == 1 ? (unit & 1 ? 0 : 1) : NC / 2; }
    static constexpr bool loads_w(int unit) { return !W4 || !(unit & 1); }
    static constexpr int items(int unit) { return copies(unit) + (loads_w(unit) ? NW : 0); }
    static constexpr int per_step() { return items(0) + (U == 2 ? items(1) : 0); }
    // loads of a wave that may be outstanding at the wait of unit `u` of a step (int4: 1)
    static constexpr int in_flight(int u) {
        int weights = 0;                                        // issued since the next weights
        if (W4) weights = items(1) + (NSW - 2) * per_step();
        else for (int t = 0; t < NSW - 2; ++t) weights += items(U == 1 ? 0 : (u + t) & 1);
        // issued since the last copy of step B + G + 1 - D
        const int copied = (W4 ? (NC == 1 ? NW : 0) : U == 2 && NC == 1 ? 2 * NW : NW) + (D - G - 1) * per_step();
        return u == U - 1 && copied < weights ? copied : weights;
    }
    // weights loaded in `unit`: of which unit (int4: step)
    static constexpr int loaded(int unit) { return W4 ? (unit >> 1) + NSW - 1 : unit + NSW - 1; }
    // what the prologue has issued since the last of what the first unit and the reads up to the first barrier need: the
    // weights of unit 0 and the copies of steps 0 .. G
    static constexpr int prologue_since() {
        int n = 0, last = 0;
        for (int t = 0; t < U * D; ++t) {
            n += copies(t % U);
            if (t / U <= G) last = n;
            if (loads_w(t % U) && loaded(t - U * D) >= 0) n += NW;
            if (loads_w(t % U) && loaded(t - U * D) == 0) last = n;
        }
        return n - last;
    }
    static_assert(D >= G + 1 && NBUF >= D + G && UNR % G == 0 && (W4 ? UNR : U * UNR) % NSW == 0, "see the ordering rules above");
    static_assert(in_flight(0) <= 63 && in_flight(U - 1) <= 63, "the vmcnt field");
    static_assert(NBUF * BUF <= WK_RING_BYTES && 4 * RM * CN * 1024 <= WK_RING_BYTES, "the ring; the exchange of k-halves");
};

// Where a load is issued: the wave's priority there and the step of the trip, -1 in the prologue.
template <int P, int STEP> struct WkAt { static constexpr int PRIO = P, AT = STEP; };
// The tiles that a workgroup of gemm_wk_big_kernel multiplies one after the other: v, v + stride, .. below `big`.
struct WkChain { int v, stride, big, mblocks, nblocks; };

// RAW: the activations are the caller's int8 rows (g.A_rows, rows and K of 16-byte pieces), not tiles of them.  A copy then brings whole
// 128-byte lines, 4 or 8 rows of one step; piece p of a row lies in slot p ^ swizzle(row) of the row's 16 or 8, so that the 16
// rows of an operand, which are a multiple of 128 bytes apart, are read from 16 different places.  The tiles that the call owes its
// caller (g.A) are written by the workgroups of a row block together, up to RAW_TILES per wave: fetched behind the
// prologue, stored behind the loop.  Without the re-tiling launch in front, us: exact
// 128 x 4096 x 11008 13.6 -> 11.8, 512 x 4096 x 4096 15.3 -> 12.8, 1000 x 2048 x 4096 15.4 -> 13.1, 300 x 14336 x 4096 38.2 -> 33.6 (and 11.6, 13.0,
// 12.4 and 33.5 since the k-halves meet in branches and the zeros are written early, another box).
constexpr int RAW_TILES = 4;

template <int TM, bool W4, int EPI, int TN, bool RS, bool RAW = false>
__device__ __forceinline__ void wk_tile(const rkh_gemm_args& g, uint8_t* lds_raw, int tile, int mblk, int nblk, int kpart,
                                        int ksplit, int kt0, int kts, // the part's first k-tile and their number, a multiple of 8
                                        [[maybe_unused]] WkChain chain = {}) {
    using S = WkShape<TM, W4, TN, RS>;
    static_assert(!RAW || (!RS && !W4 && EPI == RKH_EPI_I32 && S::NC == 2), "int8 rows as given: the exact product on narrow tiles");
    static_assert(TN == 2 || (TN == 1 && EPI != RKH_EPI_SWIGLU), "gate / up pairs need two column blocks per wave");
    constexpr int U = S::U, RM = S::RM, CN = S::CN, KT = S::KT, BUF = S::BUF, NBUF = S::NBUF, NSW = S::NSW;
    constexpr int A_STEP = RAW ? KT * 32 : KT * 1024, W_STEP = KT * (W4 ? 512 : 1024);

    const int lane = lane_id();
    const int wave = __builtin_amdgcn_readfirstlane(wave_id());
    const int wn = wave & 3, wk = wave >> 2; // column group; k-half (RS: row half)
    const int KB = (int)rkh_align_up(g.K, RKH_K_ALIGN) / 32;

    // ---- sources: wave-uniform base pointers (scalar registers) + a constant lane offset.
    // The step's copies of a wave are NC consecutive KiB: of row block wave * NC / KT, from k-tile wave * NC % KT on
    const auto a_from = [&](int mb) { return g.A + ((size_t)(mb * (S::BM / 32) + wave * S::NC / KT) * KB + kt0 + wave * S::NC % KT) * 1024; };
    const auto w_from = [&](int nb, int j) { // (int4: two k-tiles per KiB)
        return g.W + ((size_t)(nb * (4 * TN) + wn * TN + j) * KB + kt0 + (RS ? 0 : wk * 2 * U)) * (W4 ? 512 : 1024);
    };
    const uint8_t* asrc = RAW ? g.A_rows + (size_t)(mblk * S::BM) * g.K : a_from(mblk);
    const uint8_t* wsrc[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) wsrc[j] = w_from(nblk, j);
    const int q = lane >> 4;
    const unsigned lane_off = lane * 16;
    const unsigned piece_off = (q >> 1) * 1024 + (q & 1) * 512 + (lane & 15) * 16; // this lane's piece of an operand
    const uint32_t lds_base = (uint32_t)(uintptr_t)(lds_ptr_t)lds_raw;
    uint32_t copy_lo = lds_base + wave * S::NC * 1024, copy_hi = copy_lo + 65536; // this wave's chunk inside buffer 0, and 64 KiB on
    // LDS byte addresses of this lane's piece of the wave's first operand in buffer 0 and 64 KiB on
    uint32_t frag_lo = lds_base + (RS ? wk * (RM / 2) * KT : wk * 2 * U) * 1024 + (W4 ? piece_off + (q >> 1) * 1024 : piece_off);
    uint32_t frag_hi = frag_lo + 65536;
    const int ksteps = kts / KT;
    // RAW: this lane's places in the rows of the step's two copies, the same for the step that K ends in (pieces beyond K: the row's
    // first, any would do -- the weights there are zero), and its first piece of the operands of each unit of a step
    constexpr int PIECES = KT * 2, COPY_ROWS = 64 / PIECES, SWIZZLE = PIECES == 16 ? 0 : 1; // swizzle(row) = row >> SWIZZLE, modulo PIECES
    [[maybe_unused]] unsigned row_off[2], row_off_end[2];
    [[maybe_unused]] uint32_t raw_lo[U], raw_hi[U];
    if constexpr (RAW) {
        const unsigned in_step = (g.K - 1) % (KT * 32) + 1; // k of the last step with any
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const int row = (wave * 2 + c) * COPY_ROWS + lane / PIECES;
            const unsigned piece = ((lane % PIECES) ^ (row >> SWIZZLE)) % PIECES;
            row_off[c] = (unsigned)min(row, g.M - 1 - mblk * S::BM) * (unsigned)g.K + piece * 16;
            row_off_end[c] = piece * 16 < in_step ? row_off[c] : row_off[c] - piece * 16;
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int r = lane & 15, piece = ((wk * 4 * U + u * 4 + q) ^ (r >> SWIZZLE)) % PIECES;
            raw_lo[u] = lds_base + r * (PIECES * 16) + piece * 16;
            raw_hi[u] = raw_lo[u] + 65536;
        }
    }
    // how often the sources may still advance (RAW: rows end with K, which a step of 128 k may lie beyond)
    int a_left = (RAW ? (g.K + KT * 32 - 1) / (KT * 32) : ksteps) - 1, w_left = ksteps - 1;
    // RS: where they go from there, the chain's next tile or, behind the last, nowhere
    [[maybe_unused]] const uint8_t *a_next = nullptr, *w_next[TN] = {};
    [[maybe_unused]] int a_step = A_STEP, w_step = W_STEP, mblk_next = 0, nblk_next = 0;
    [[maybe_unused]] bool more = false, a_turn = false, w_turn = false; // a_turn, w_turn: in this trip
    [[maybe_unused]] const auto find_next = [&]() {
        more = chain.v + chain.stride < chain.big;
        if (more) wk_tile_coords(xcd_remap(chain.v + chain.stride, chain.big), chain.mblocks, chain.nblocks, mblk_next, nblk_next);
        a_next = more ? a_from(mblk_next) : a_from(mblk) + (size_t)(ksteps - 1) * A_STEP;
#pragma unroll
        for (int j = 0; j < TN; ++j) w_next[j] = more ? w_from(nblk_next, j) : w_from(nblk, j) + (size_t)(ksteps - 1) * W_STEP;
    };
    // (the prologue reaches the end of a tile only if there is no other, see launch_gemm_wk_big)
    if constexpr (RS) a_next = asrc + (size_t)(ksteps - 1) * A_STEP;

    v4i acc[RM][CN];
    v4i a[RM];                  // activation operands
    v4i wring[NSW][CN];         // weights as loaded: of a unit, or, int4, of a step
    [[maybe_unused]] v4i wop[2][CN]; // int4 only: unpacked operands, this unit / next

    // Copies beyond K are issued like the others, for the count.  Tiles of 64 x 128 with int8 weights, which are bound by
    // the compute unit's memory path, issue them for one lane: three steps of 16 KiB that nothing reads, beside the 16 of
    // K = 4096 (exact 128 x 4096 x 11008 13.9 -> 13.65 us, 512 x 4096 x 4096 16.5 -> 16.3; int4 weights and wider tiles gain nothing).
    constexpr bool MASKED = (TM == 2 && TN == 1 && !W4) || RAW;
    [[maybe_unused]] unsigned long long a_lanes = ~0ull;
    auto copy_a = [&](auto buf_tag, auto c_tag, auto at_tag) { // one of the step's copies
        constexpr int C = decltype(c_tag)::value, PRIO = decltype(at_tag)::PRIO;
        constexpr int B = decltype(buf_tag)::value % NBUF, PER = 65536 / BUF;
        const uint32_t dst = (B < PER ? copy_lo : copy_hi) + B % PER * BUF;
        if constexpr (RAW) copy_lds<0, PRIO>(a_left > 0 ? row_off[C & 1] : row_off_end[C & 1], asrc, dst + C * 1024, a_lanes);
        else if constexpr (MASKED) copy_lds<C * 1024, PRIO>(lane_off, asrc, dst, a_lanes);
        else copy_lds<C * 1024, PRIO>(lane_off, asrc, dst);
        // RS: a trip turns to the next tile behind one of its steps (a choice behind every step cost the loop 2.5 %)
        if constexpr (C == S::NC - 1 && RS && decltype(at_tag)::AT >= 0 && decltype(at_tag)::AT != S::A_TURN) {
            asrc += a_step;
        } else if constexpr (C == S::NC - 1 && RS) {
            const bool turn = decltype(at_tag)::AT < 0 ? a_left-- == 0 : a_turn;
            asrc = turn ? a_next : asrc + a_step;
            a_step = turn && !more ? 0 : a_step;
        } else if constexpr (C == S::NC - 1) {
            asrc += a_left > 0 ? A_STEP : 0;
            if constexpr (MASKED) a_lanes = a_left > 0 ? ~0ull : 1ull;
            --a_left;
        }
    };
    auto load_w = [&](v4i* regs, auto half_tag, auto e_tag, [[maybe_unused]] auto at_tag) { // operand e of unit HALF of a step (int4: of both)
        constexpr int HALF = W4 || U == 1 ? 0 : decltype(half_tag)::value, E = decltype(e_tag)::value;
        load_regs<HALF * 2048 + (E & 1) * 256>(regs[E], piece_off, wsrc[E / 2]);
        if constexpr (E == CN - 1 && RS && decltype(at_tag)::AT != S::W_TURN) {
#pragma unroll
            for (int j = 0; j < TN; ++j) wsrc[j] += w_step;
        } else if constexpr (E == CN - 1 && RS) {
#pragma unroll
            for (int j = 0; j < TN; ++j) wsrc[j] = w_turn ? w_next[j] : wsrc[j] + w_step;
            w_step = w_turn && !more ? 0 : w_step;
        } else if constexpr (E == CN - 1 && (W4 || HALF == U - 1)) {
#pragma unroll
            for (int j = 0; j < TN; ++j) wsrc[j] += w_left > 0 ? W_STEP : 0;
            --w_left;
        }
    };
    auto w_wait = [&](v4i* regs, auto n_tag) { // regs become valid
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(n_tag)::value) : "memory");
#pragma unroll
        for (int e = 0; e < CN; ++e) keep(regs[e]);
    };
    auto read_a = [&](auto unit_tag, auto i_tag) { // operand i of a unit of the trip; awaited by wait_lds
        constexpr int UNIT = decltype(unit_tag)::value, I = decltype(i_tag)::value, B = UNIT / U % NBUF, PER = 65536 / BUF;
        if constexpr (RAW) read_lds<B % PER * BUF + I * (PIECES * 256)>(a[I], B < PER ? raw_lo[UNIT % U] : raw_hi[UNIT % U]);
        else read_lds<B % PER * BUF + (I / 2) * KT * 1024 + (UNIT % U) * (W4 ? 1024 : 2048) + (I & 1) * 256>(a[I], B < PER ? frag_lo : frag_hi);
    };
    auto unpack = [&](v4i* dst, const v4i* raw, auto half_tag, auto e_tag) { // k-tile HALF of each super-tile
        if constexpr (W4) {
            constexpr int HALF = decltype(half_tag)::value, E = decltype(e_tag)::value;
            const int x = HALF ? raw[E].z : raw[E].x, y = HALF ? raw[E].w : raw[E].y;
            dst[E] = v4i{(x << 4) & (int)0xF0F0F0F0, x & (int)0xF0F0F0F0, (y << 4) & (int)0xF0F0F0F0, y & (int)0xF0F0F0F0};
            if constexpr (S::ASM) keep(dst[E]); // (here, not in front of the product, see mfma())
        }
    };

    // Unit t of the trip.  FRESH: the accumulators start here.
    auto k_unit = [&](auto unit_tag, auto fresh_tag) {
        constexpr int T = decltype(unit_tag)::value, STEP = T / U, UN = T % U, MF = RM * CN;
        constexpr int ITEMS = S::items(UN), LAST = W4 ? MF / 2 : MF, SPACE = LAST / (ITEMS + 1) > 0 ? LAST / (ITEMS + 1) : 1; // loads: behind every SPACE-th MFMA
        static_assert(ITEMS * SPACE <= (W4 && UN == 0 ? MF : LAST), "every load of a unit goes out before its wait");
        constexpr int NEXT_W = W4 ? (STEP + 1) % NSW : (T + 1) % NSW;                 // slot of the next unit's (step's) weights
        constexpr int LOAD_SLOT = W4 ? (STEP + NSW - 1) % NSW : (T + NSW - 1) % NSW;
        using Half = std::integral_constant<int, (T + NSW - 1) & 1>;                  // place in its step of the unit whose weights are loaded
        // The two waves of a SIMD drift apart between barriers (the older one wins every issue conflict) and the one left
        // behind cannot keep the matrix pipe busy alone: the wave that is further into the barrier interval yields.
        // (4096 x 4096 x 14336 int8 185.4 -> 182.7 us, 200 x 4096 x 14336 int4 18.1 -> 17.5)
        using At = WkAt<3 - 4 * (T % (U * S::G)) / (U * S::G), STEP>;
        static_for<RM>([&](auto i_tag) {
            constexpr int I = decltype(i_tag)::value;
            wait_lds<RM - 1, !S::ASM>(a[I]);
            static_for<CN>([&](auto j_tag) {
                constexpr int J0 = decltype(j_tag)::value, J = I & 1 ? CN - 1 - J0 : J0, AT = I * CN + J0; // (there and back: one operand stays)
                const v4i& w = W4 ? wop[UN][J] : wring[T % NSW][J];
                if constexpr (!S::ASM) acc[I][J] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w, a[I], acc[I][J], 0, 0, 0);
                else if constexpr (decltype(fresh_tag)::value && T == 0) mfma_first(acc[I][J], w, a[I]);
                else mfma(acc[I][J], w, a[I]);
                if constexpr (AT % SPACE == SPACE - 1 && AT / SPACE < ITEMS) {
                    constexpr int Q = AT / SPACE, NCU = S::copies(UN);
                    if constexpr (Q < NCU) copy_a(std::integral_constant<int, STEP + S::D>{}, std::integral_constant<int, Q + (UN ? S::copies(0) : 0)>{}, At{});
                    else load_w(wring[LOAD_SLOT], Half{}, std::integral_constant<int, Q - NCU>{}, At{});
                }
                if constexpr (W4) { // the next unit's operands, in the second half of this one
                    if constexpr (UN == 1 && AT == MF / 2 - 1) w_wait(wring[NEXT_W], std::integral_constant<int, S::in_flight(1)>{});
                    constexpr int EVERY = MF / 2 / CN, K = AT - MF / 2;
                    if constexpr (K >= 0 && K % EVERY == 0)
                        unpack(wop[UN ^ 1], wring[UN ? NEXT_W : STEP % NSW], std::integral_constant<int, UN ^ 1>{}, std::integral_constant<int, K / EVERY>{});
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            read_a(std::integral_constant<int, T + 1>{}, i_tag);
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (!W4) w_wait(wring[NEXT_W], std::integral_constant<int, S::in_flight(UN)>{});
        if constexpr (UN == U - 1 && (STEP + 1) % S::G == 0) asm volatile("s_barrier" ::: "memory");
    };
    auto k_step = [&](auto step_tag, auto fresh_tag) {
        static_for<U>([&](auto u_tag) { k_unit(std::integral_constant<int, U * decltype(step_tag)::value + decltype(u_tag)::value>{}, fresh_tag); });
    };

    // prologue: the same issue order as if the loop had run for steps -D..-1
    static_for<U * S::D>([&](auto t_tag) {
        constexpr int T = decltype(t_tag)::value - U * S::D, UN = (T + U * S::D) % U, OF = S::loaded(T);
        static_for<S::copies(UN)>([&](auto c_tag) {
            copy_a(std::integral_constant<int, (T + U * S::D) / U>{}, std::integral_constant<int, decltype(c_tag)::value + (UN ? S::copies(0) : 0)>{}, WkAt<0, -1>{});
        });
        if constexpr (S::loads_w(T) && OF >= 0)
            static_for<CN>([&](auto e_tag) { load_w(wring[OF % NSW], std::integral_constant<int, OF & 1>{}, e_tag, WkAt<0, -1>{}); });
    });
    RK_TS(1);
    // The tile's scales follow, straight to LDS, so that the epilogue does not start with a round trip to memory: thread t
    // brings the scale of row t % BM and of physical column t % (128 TN).  (Two more loads in the queue only make the
    // first units' waits stricter.  Ahead of the prologue's loads they cost the 128-row tile 0.2 us: the first copies
    // leave later.  Rows and columns beyond the matrix take some valid scale: nothing is stored for them.)
    const auto fetch_scales = [&](uint32_t to) {
        if constexpr (EPI != RKH_EPI_I32) {
            int t = threadIdx.x;
            asm volatile("" : "+v"(t)); // (opaque: addresses made from it are not worth registers in the loop)
            const int row = t & (S::BM - 1), col = t & (128 * TN - 1);
            const int pb = nblk * (4 * TN) + (col >> 5);
            const int n = EPI == RKH_EPI_SWIGLU && (pb >> 1) * 32 >= g.interleave_F ? 0 : block_first_col(pb, g.interleave_F) + (col & 31);
            copy_lds_dword(g.a_scale + min(mblk * S::BM + row, g.M - 1), lds_base + to + (wave * 64 & (S::BM - 1)) * 4);
            copy_lds_dword(g.w_scale + min(n, g.N - 1), lds_base + to + (WK_ROW_SCALES + (wave * 64 & (128 * TN - 1))) * 4);
        }
    };
    fetch_scales(WK_SCALES_OFF);
    // RAW: this wave's tiles of the caller's copy, tile `kb` of the row block `rb` of this workgroup's rows
    [[maybe_unused]] v4i copied[RAW_TILES];
    [[maybe_unused]] const int raw_all = S::BM / 32 * KB, raw_nb = (g.N + 128 * TN - 1) / (128 * TN), raw_per = (raw_all + raw_nb - 1) / raw_nb;
    [[maybe_unused]] const bool raw_many = RAW && raw_per > 8; // (more than one per wave; loads that bring nothing cost 0.3 us)
    [[maybe_unused]] const auto raw_tile = [&](int t, auto&& f) { // f(source, destination) for this lane's 16 bytes if there are any
        const int mine = wave + 8 * t, tile_of = nblk * raw_per + mine;
        const int rb = tile_of / KB, kb = tile_of - rb * KB, m = mblk * S::BM + rb * 32 + (lane & 31), k = kb * 32 + (lane >> 5) * 16;
        if (mine < raw_per && tile_of < raw_all && m < g.M && k < g.K)
            f(g.A_rows + (size_t)m * g.K + k, const_cast<uint8_t*>(g.A) + ((size_t)(mblk * (S::BM / 32) + rb) * KB + kb) * 1024 + lane * 16);
    };
    [[maybe_unused]] const auto raw_fetch = [&](int t) {
        const uint8_t* from = g.A_rows; // (every lane loads, for the count)
        raw_tile(t, [&](const uint8_t* src, uint8_t*) { from = src; });
        load_far(copied[t], from);
    };
    if constexpr (RS) find_next(); // (while the first loads are on their way)
    if constexpr (RAW) {
        raw_fetch(0);
        if (raw_many) {
#pragma unroll
            for (int t = 1; t < RAW_TILES; ++t) raw_fetch(t);
        }
    }
    // The sums' zeros, while the first loads are on their way.  Named, so that they are written here: the compiler wrote them
    // behind the wait for the first data, and of a workgroup's small tiles it kept zeros in scratch memory, whose loads
    // and stores wait among the prologue's.  us: int8 4000 x 1024 x 14336 73.8 -> 72.7, 786 x 661 x 8720 18.9 -> 18.5, 505 x 544 x 8320 12.8 ->
    // 12.7, int4 2156 x 640 x 2176 13.8 -> 13.6, exact 4007 x 1024 x 9088 58.7 -> 57.5, the FFN 1300 x 512 x 12288 95.2 -> 91.9.
    if constexpr (!RS) {
#pragma unroll
        for (int t = 0; t < RM * CN; ++t) {
            acc[t / CN][t % CN] = v4i{0, 0, 0, 0};
            keep(acc[t / CN][t % CN]);
        }
    }
    // weights of unit 0 and the copies of steps 0..G land (RAW: one load or RAW_TILES behind them, the count of one)
    w_wait(wring[0], std::integral_constant<int, S::prologue_since() + (EPI != RKH_EPI_I32 ? 2 : 0) + (RAW ? 1 : 0)>{});
    asm volatile("s_barrier" ::: "memory");
    const auto first_operands = [&]() {
        static_for<RM>([&](auto i_tag) { read_a(std::integral_constant<int, 0>{}, i_tag); });
        static_for<CN>([&](auto e_tag) { unpack(wop[0], wring[0], std::integral_constant<int, 0>{}, e_tag); });
    };
    first_operands();
    RK_TS(2);

    using Old = std::false_type;
    // Scale, convert and store the rows from row0 of the tile on
    const auto store = [&](auto rows_tag, auto&& sum_of, int row0, int scales) {
        constexpr int ROWS = decltype(rows_tag)::value;
        int l = lane; // (opaque, as in fetch_scales)
        asm volatile("" : "+v"(l));
        const float* sc = reinterpret_cast<const float*>(lds_raw + scales);
        float as[ROWS];
        v4f ws[CN];
        if constexpr (EPI != RKH_EPI_I32) {
#pragma unroll
            for (int i = 0; i < ROWS; ++i) as[i] = sc[row0 + i * 16 + (l & 15)];
#pragma unroll
            for (int j = 0; j < CN; ++j) ws[j] = *reinterpret_cast<const v4f*>(sc + WK_ROW_SCALES + (wn * CN + j) * 16 + 4 * (l >> 4));
        }
        wk_store<ROWS, CN, W4, EPI>(g, sum_of, [&](int i) { return as[i]; }, [&](int j, int e) { return ws[j][e]; },
                                    mblk * S::BM + row0, nblk * (4 * TN) + wn * TN, g.M, lds_raw + WK_STAGE_OFF + wave * WK_STAGE, l);
    };
    const auto settle = [&]() { // the operands that were read beyond the tile's last unit; see below for why they are named
        __builtin_amdgcn_s_setprio(0);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_nop 7\n\ts_nop 7" ::: "memory");
#pragma unroll
        for (int i = 0; i < RM; ++i) keep(a[i]);
#pragma unroll
        for (int t = 0; t < RM * CN; ++t) keep(acc[t / CN][t % CN]);
    };
    if constexpr (RS) {
        // The steps of the chain's tiles follow one another: the copies and weights that run ahead of a tile's end are the
        // next tile's first ones, and stay in the ring and in registers while the tile is converted and stored.
        for (int scales = WK_SCALES_OFF;; scales ^= WK_SCALES_OFF ^ (WK_SCALES_OFF + WK_SCALES)) {
            const auto trip = [&](auto fresh_tag, int k) {
                a_turn = k + 2 * S::UNR == ksteps, w_turn = k + S::UNR == ksteps;
                static_for<S::UNR>([&](auto step) { k_step(step, fresh_tag); });
                const uint32_t f = frag_lo, c = copy_lo;
                frag_lo = frag_hi, frag_hi = f, copy_lo = copy_hi, copy_hi = c;
            };
            trip(std::true_type{}, 0);
            for (int k = S::UNR; k < ksteps; k += S::UNR) trip(Old{}, k);
            RK_TS(3);
            settle();
            // behind the last tile: a load to LDS must not outlive the workgroup (waited for here, not behind the stores)
            if (!more) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            RK_TS(4);
            store(std::integral_constant<int, RM>{}, [&](int i, int j) -> const v4i& { return acc[i][j]; }, wk * RM * 16, scales);
            RK_TS(5);
            if (!more) break;
            chain.v += chain.stride;
            mblk = mblk_next, nblk = nblk_next;
            find_next();
            fetch_scales(scales ^ WK_SCALES_OFF ^ (WK_SCALES_OFF + WK_SCALES));
            first_operands();
        }
        return;
    }

    int s = 0;
    for (; s + S::UNR <= ksteps; s += S::UNR) static_for<S::UNR>([&](auto step) { k_step(step, Old{}); });
    // (the remaining steps as a chain that ends at the first one beyond K: the control flow
    // then only holds the sequences of steps that can happen, which is what the static check
    // of the waits, audit_waits.py, walks)
    static_while<S::UNR - 1>([&](auto step) {
        if (s + decltype(step)::value >= ksteps) return false;
        k_step(step, Old{});
        return true;
    });
    RK_TS(3);

    // ---- epilogue.  Drain the look-ahead copies (they write LDS), the operands read ahead and the scale
    // loads; then every wave is past its last operand and LDS is reused.
    settle();
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    // What was loaded for units beyond K was in flight until this wait, while the compiler regards
    // the destination registers as dead: the uses below keep it from giving one of them to an epilogue value
    // ahead of the wait (the load would then land on top of that value).
#pragma unroll
    for (int t = 0; t < NSW; ++t)
#pragma unroll
        for (int e = 0; e < CN; ++e) keep(wring[t][e]);
    if constexpr (RAW) {
        const auto raw_store = [&](int t) {
            keep(copied[t]);
            raw_tile(t, [&](const uint8_t*, uint8_t* dst) { *reinterpret_cast<v4i*>(dst) = copied[t]; });
        };
        raw_store(0);
        if (raw_many) {
#pragma unroll
            for (int t = 1; t < RAW_TILES; ++t) raw_store(t);
        }
    }
    lds_barrier();

    // The k-halves meet: a wave hands half of the rows of its strip to its partner and keeps operands wk * RM / 2 ..
    // Accumulators are indexed with constants, hence the two branches.
    if constexpr (!RS) {
        constexpr int KEEP = RM / 2, XT = KEEP * CN; // operands kept; tiles per exchange slot
        v4i sum[KEEP][CN];
        v4i* xch = reinterpret_cast<v4i*>(lds_raw);
        // (The comment at the end, which differs between the two branches, keeps the compiler from making one of them: it
        // would select each accumulator with a vector instruction, 128 in a tile of 128 x 256.  From the loop to the
        // first store 2.1 -> 1.5 us; calls, us: int4 2048 x 512 x 4096 14.2 -> 13.3, 4036 x 640 x 1920 19.1 -> 18.1, int8 786 x 661 x 8720
        // 18.1 -> 17.3, exact 950 x 1408 x 5120 15.9 -> 15.4, the FFN 188 x 4576 x 11584 57.0 -> 55.3.)
        const auto meet = [&](auto wk_tag) {
            constexpr int GIVE0 = (decltype(wk_tag)::value ^ 1) * KEEP, KEEP0 = decltype(wk_tag)::value * KEEP;
#pragma unroll
            for (int t = 0; t < XT; ++t) xch[(wave * XT + t) * 64 + lane] = acc[GIVE0 + t / CN][t % CN];
            lds_barrier();
#pragma unroll
            for (int t = 0; t < XT; ++t) sum[t / CN][t % CN] = acc[KEEP0 + t / CN][t % CN] + xch[((wave ^ 4) * XT + t) * 64 + lane];
            asm volatile("; rows of k-half %0" ::"n"(KEEP0));
        };
        if (wk == 0) meet(std::integral_constant<int, 0>{});
        else meet(std::integral_constant<int, 1>{});
        if (ksplit > 1) { // partial tile in accumulator order: [tile][part][wave][kept tile][lane] x 4 ints
            v4i* dst = reinterpret_cast<v4i*>(g.splitk_acc) + (((size_t)tile * ksplit + kpart) * 8 + wave) * (XT * 64);
#pragma unroll
            for (int t = 0; t < XT; ++t) dst[t * 64 + lane] = sum[t / CN][t % CN];
            return;
        }
        RK_TS(4);
        store(std::integral_constant<int, KEEP>{}, [&](int i, int j) -> const v4i& { return sum[i][j]; }, wk * KEEP * 16, WK_SCALES_OFF);
        RK_TS(5);
    }
}

// The tile of a workgroup: XCD-contiguous ranges, 4 row blocks per column sweep.
template <int TM, bool W4, int EPI, int TN = 2, bool RAW = false>
__global__ __launch_bounds__(512) void gemm_wk_kernel(const uint8_t* h_A, const uint8_t* h_W, int h_M, int h_K,
                                                      int mblocks, int nblocks, int ksplit, int units_per_part,
                                                      rkh_gemm_args g) {
    // (leading scalar arguments, see RK_GEMM_HEAD_PARAMS: everything the tile coordinates and the
    // prologue's loads depend on, ten dwords, arrives in registers)
    g.A = h_A; g.W = h_W; g.M = h_M; g.K = h_K;
    RK_TS(0);
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[]; // WK_LDS_BYTES
    const int units = (int)rkh_align_up(g.K, RKH_K_ALIGN) / WK_PART_K;
    const int tiles = mblocks * nblocks;
    const int logical = xcd_remap(blockIdx.x, tiles * ksplit);
    const int kpart = ksplit > 1 ? (int)((unsigned)logical / (unsigned)tiles) : 0;
    const int tile = logical - kpart * tiles;
    int mblk, nblk;
    wk_tile_coords(tile, mblocks, nblocks, mblk, nblk);
    const int first = kpart * units_per_part; // (at least one unit by construction of the launch)
    wk_tile<TM, W4, EPI, TN, false, RAW>(g, lds_raw, tile, mblk, nblk, kpart, ksplit, first * (WK_PART_K / 32),
                                    min(units_per_part, units - first) * (WK_PART_K / 32));
}

// Tiles of 256 x 256 (RS) -- `big` of them, the first in tile order -- and tiles of 128 x 256 for what is
// left of the output: the tiles that would start a last, mostly empty round, each in two halves, and a
// last strip of at most 128 rows.  Workgroup = 8 waves in 4 column groups x 2 row halves: a wave multiplies
// 128 x 64 over the whole K, so there is no exchange of k-halves and all eight waves convert and store.
// What bounds it: the matrix pipes at the clock that the power limit leaves, and the conversion and stores of a tile.
// A workgroup per compute unit multiplies its tiles one after the other as one stream of steps (wk_tile, RS), so that the first
// operands of every tile but its first are in LDS and registers when the tile before has been stored (its first wait for
// weights, two units later, stands behind that tile's 16 or 32 stores, which the counter counts too): int8 4000 x 1024 x 14336
// 77.9 -> 73.2 us, 4000 x 512 x 14336 67.3 -> 62.4, 4096 x 4096 x 14336 187 -> 184; a launch of one round measures the same.  The small tiles behind a chain
// start with a round trip to memory each.
// Against 128 x 256 tiles: the second operand of a column group comes once per 256 rows (16 instead of 24 KB from L2 per 512
// cycles of MFMAs), one prologue and one epilogue per 256 rows.  us, quantization included, when the tiles were
// introduced: int8 4096 x 4096 x 14336 241 -> 203, 2048 x 4096 x 14336 122 -> 108, 4096^3 74.7 -> 68.1; int4 214 -> 195, 75 -> 69.
// (Measured and not kept: half of the compute units starting with a small tile so that the epilogues'
// bursts of stores fall apart -- 204 -> 217, 195 -> 210: tiles in step share their operands in L2.)
template <bool W4, int EPI>
__global__ __launch_bounds__(512) void gemm_wk_big_kernel(const uint8_t* h_A, const uint8_t* h_W, int h_M, int h_K,
                                                          int mblocks, int nblocks, int big, int small, int rounds, rkh_gemm_args g) {
    g.A = h_A; g.W = h_W; g.M = h_M; g.K = h_K;
    RK_TS(0);
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_raw[]; // WK_LDS_BYTES
    const int KB = (int)rkh_align_up(g.K, RKH_K_ALIGN) / 32;
    const int groups = gridDim.x, b = blockIdx.x;
    int mblk, nblk;
    if (b < big) {
        wk_tile_coords(xcd_remap(b, big), mblocks, nblocks, mblk, nblk);
        wk_tile<4, W4, EPI, 2, true>(g, lds_raw, 0, mblk, nblk, 0, 1, 0, KB, WkChain{b, groups, big, mblocks, nblocks});
    }
    // The small tiles: `rounds` for every workgroup without a big one in the last round, the rest for the others.  (Without
    // rounds -- a workgroup per tile -- they follow the big ones.)
    const int extra = rounds ? big % groups : big, without = groups - extra;
    const int first = b >= extra ? b - extra : without * rounds + b, stride = b >= extra ? without : extra;
    const int end = !rounds ? b >= extra ? first + 1 : 0 : b >= extra ? min(small, without * rounds) : small;
    const int halves = 2 * (mblocks * nblocks - big); // small tiles inside the last 256 x 256 ones, then the strip
    if (first < end) asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // (no load is in flight, but only the chain's loop knows that)
    for (int s = first; s < end; s += stride) {
        lds_barrier(); // every wave is past the tile before: the ring and the staging areas are free
        const int t = xcd_remap(s, small);
        if (t < halves) {
            wk_tile_coords(big + (t >> 1), mblocks, nblocks, mblk, nblk);
            mblk = mblk * 2 + (t & 1);
        } else {
            mblk = mblocks * 2;
            nblk = t - halves;
        }
        wk_tile<4, W4, EPI, 2, false>(g, lds_raw, 0, mblk, nblk, 0, 1, 0, KB);
    }
}

// Second half of a K-split launch.  Workgroup = one wave = up to 32 rows of what one wave of gemm_wk_kernel kept of an output
// tile: blockIdx.x = (tile * 8 + wave) * PARTS + part.  Adds the ksplit partial tiles and runs the epilogue.  Bound by the latency
// of its loads, which a wave has in flight for one part of K at a time: the loads of a part go out together (left to itself the
// compiler waited for each of them ahead of the next in the exact product of 128-row tiles), and the 64 rows that a wave of
// the 128-row tile kept go to two waves.  us, one wave with loads as the compiler had them -> loads together -> two
// waves: exact 737 x 10240 x 700 29.7 -> 25.1 -> 24.1, 2076 x 10240 x 512 35.8 -> 33.9 -> 33.2, 453 x 8733 x 628 (64-row tiles) 25.4 ->
// 24.1, int8 737 x 10240 x 700 30.0 -> 29.7 -> 27.6, 1135 x 8960 x 2176 42.8 -> 43.0 -> 42.0.
template <int TM, bool W4, int EPI>
__global__ __launch_bounds__(64) void gemm_wk_reduce_kernel(rkh_gemm_args g, int mblocks, int nblocks, int ksplit) {
    constexpr int TN = 2, CN = 4, BM = 32 * TM, KEEP = TM; // (operands of 16 rows that a wave kept)
    constexpr int ROWS = KEEP > 2 ? 2 : KEEP, PARTS = KEEP / ROWS;
    __shared__ __attribute__((aligned(16))) uint8_t stage_lds[WK_STAGE];
    const int lane = lane_id();
    const int owner = blockIdx.x / PARTS, part = blockIdx.x % PARTS;
    const int tile = owner / 8, wave = owner % 8, wn = wave & 3, wk = wave >> 2;
    int mblk, nblk;
    wk_tile_coords(tile, mblocks, nblocks, mblk, nblk);
    const int m0 = mblk * BM + (wk * KEEP + part * ROWS) * 16, pb0 = nblk * 8 + wn * TN;
    const v4i* src = reinterpret_cast<const v4i*>(g.splitk_acc) + ((size_t)tile * ksplit * 8 + wave) * (KEEP * CN * 64) + part * (ROWS * CN * 64) + lane;
    v4i sum[ROWS][CN];
#pragma unroll
    for (int t = 0; t < ROWS * CN; ++t) sum[t / CN][t % CN] = v4i{0, 0, 0, 0};
    for (int p = 0; p < ksplit; ++p, src += 8 * KEEP * CN * 64) {
        // int4 weights ride as 16 * code: a part's sum is an exact multiple of 16 that fits
        // int32 (a part spans at most 2^17 k), but the sum of the parts times 16 need not --
        // so the factor comes off each part before it is added
        v4i got[ROWS * CN];
#pragma unroll
        for (int t = 0; t < ROWS * CN; ++t) got[t] = src[t * 64];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < ROWS * CN; ++t) sum[t / CN][t % CN] += got[t] >> (W4 ? 4 : 0);
    }
    float as[ROWS], ws[CN][4];
    if constexpr (EPI != RKH_EPI_I32) {
#pragma unroll
        for (int i = 0; i < ROWS; ++i) {
            const int m = m0 + 16 * i + (lane & 15);
            as[i] = m < g.M ? g.a_scale[m] : 0.0f;
        }
#pragma unroll
        for (int j = 0; j < CN; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int pb = pb0 + j / 2, n = block_first_col(pb, g.interleave_F) + 16 * (j & 1) + 4 * (lane >> 4) + e;
                const bool live = g.interleave_F ? pb < g.N / 32 : n < g.N;
                ws[j][e] = live ? g.w_scale[n] : 0.0f;
            }
    }
    wk_store<ROWS, CN, false, EPI>(g, [&](int i, int j) -> const v4i& { return sum[i][j]; }, [&](int i) { return as[i]; },
                                   [&](int j, int e) { return ws[j][e]; }, m0, pb0, g.M, stage_lds, lane);
}

// Bytes of split-K scratch for `tiles` output tiles of bm rows split into
// ksplit parts: the int32 partial tiles.
static size_t wk_scratch_bytes(long tiles, int bm, int ksplit) {
    return ksplit > 1 ? (size_t)tiles * ksplit * bm * 256 * 4 : 0;
}

// Workgroups of a launch with this tile height and K split (what launch_gemm_wk makes of `ksplit`).
static int wk_grid(const rkh_gemm_args& g, int tile_rows, int& ksplit) {
    const int mblocks = (g.M + tile_rows - 1) / tile_rows, nblocks = (g.N + 255) / 256;
    const int units = (int)(rkh_align_up(g.K, RKH_K_ALIGN) / WK_PART_K);
    if (ksplit > units) ksplit = units;
    if (ksplit < 1) ksplit = 1;
    const int per = (units + ksplit - 1) / ksplit;
    ksplit = (units + per - 1) / per; // no empty part
    return mblocks * nblocks * ksplit;
}

template <int TM>
int launch_gemm_wk(hipStream_t st, const rkh_gemm_args& g, int ksplit) {
    constexpr int BM = 32 * TM;
    const int mblocks = (g.M + BM - 1) / BM;
    const int nblocks = (g.N + 255) / 256;
    const int units = (int)(rkh_align_up(g.K, RKH_K_ALIGN) / WK_PART_K);
    const dim3 grid(wk_grid(g, BM, ksplit)), block(512);
    const int per = (units + ksplit - 1) / ksplit;
    mark(st, "gemm_wk_kernel");
#define RK_WK(W4, EPI)                                                                              \
    do {                                                                                            \
        /* the LDS opt-in is per function and per device: once for each device this process uses */ \
        /* (several threads may get here together: setting the attribute twice is harmless, and the  \
           flag is only set once a call has succeeded) */                                           \
        static std::atomic<bool> opted_in[64] = {};                                                 \
        int dev = 0;                                                                                \
        RKH_CHECK(hipGetDevice(&dev));                                                              \
        if (dev < 0 || dev >= 64) return RKH_ERR_RUNTIME;                                           \
        if (!opted_in[dev].load(std::memory_order_acquire)) {                                       \
            RKH_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_wk_kernel<TM, W4, EPI>), \
                                          hipFuncAttributeMaxDynamicSharedMemorySize, WK_LDS_BYTES)); \
            opted_in[dev].store(true, std::memory_order_release);                                   \
        }                                                                                           \
        hipLaunchKernelGGL((gemm_wk_kernel<TM, W4, EPI>), grid, block, WK_LDS_BYTES, st,           \
                           g.A, g.W, g.M, g.K, mblocks, nblocks, ksplit, per, g);                   \
        if (ksplit > 1) mark(st, "gemm_wk_reduce_kernel");                                          \
        if (ksplit > 1)                                                                             \
            hipLaunchKernelGGL((gemm_wk_reduce_kernel<TM, W4, EPI>),                                \
                               dim3(mblocks * nblocks * 8 * (TM > 2 ? TM / 2 : 1)), dim3(64), 0, st, g, \
                               mblocks, nblocks, ksplit);                                           \
    } while (0)
    // (a dense SwiGLU GEMM exists for int4 weights only: the w4a8 FFN; the MoE layer's is grouped)
    switch (g.epilogue) {
    case RKH_EPI_I32: if (g.w_int4) RK_WK(true, RKH_EPI_I32); else RK_WK(false, RKH_EPI_I32); break;
    case RKH_EPI_F16: if (g.w_int4) RK_WK(true, RKH_EPI_F16); else RK_WK(false, RKH_EPI_F16); break;
    case RKH_EPI_F32: if (g.w_int4) RK_WK(true, RKH_EPI_F32); else RK_WK(false, RKH_EPI_F32); break;
    case RKH_EPI_SWIGLU: if (g.w_int4) RK_WK(true, RKH_EPI_SWIGLU); else return RKH_ERR_RUNTIME; break;
    default: return RKH_ERR_RUNTIME;
    }
#undef RK_WK
    RKH_CHECK(hipGetLastError());
    return RKH_OK;
}

// How a dense launch is cut into 256 x 256 tiles (the first `big`, in tile order) and 128 x 256 ones, and
// the microseconds to expect.  A 256 x 256 tile costs 9 us beside its loop, a 128 x 256 one 8 (time stamps of tiles that were
// a workgroup each: prologue 2.5, epilogue and stores 5 - 6, the next workgroup's start 0.6), so one big tile is cheaper
// than two small ones (K = 4096: 58 against 2 x 33 us, int8 weights) but leaves more compute units idle in
// the last round: the tiles of that round go as halves where that ends sooner.
// The model is older than the kernels: every tile of a chain is charged the start that only the first one has, and the loop's
// times are those of 32x32x32 products.  Against forced plans (128 / 64 / 32-row tiles, one and two parts of K, narrow tiles) on
// 46 shapes of 64 - 4096 rows, int8, int4 and exact results, the dispatch as a whole is fastest or within 1 % on 43; behind by 3.0 %
// at int4 400 x 14336 x 2048 (narrow tiles), 5.6 % at int8 3000 x 1024 x 9000 (128 x 128 tiles), 16 % at exact 300 x 4096 x 11008 (128 x 256).
// (A forced 256:1 is cut by this function too, so the cut itself is compared with nothing.)
// `rounds`: small tiles that a compute unit without one of the last round's big tiles multiplies; the rest go to the others.
struct BigPlan { int big, small, rounds; double us, us_128; };
static BigPlan big_plan(int M, int N, int K, int w_int4) {
    const int cus = compute_units() > 0 ? compute_units() : 256;
    const int nblocks = (N + 255) / 256, strip = M % 256 > 0 && M % 256 <= 128;
    const int tiles = (M / 256 + (M % 256 > 128)) * nblocks;
    // microseconds per 64 k of a 128 x 256 tile with every compute unit at work, at the clock that the power limit leaves
    // (32x32x32 products, a tenth longer than now)
    const double loop = (w_int4 ? 0.35 : 0.39) * (rkh_align_up(K, RKH_K_ALIGN) / 64);
    const double t_big = 2 * loop + 9.0, t_small = loop + 8.0;
    BigPlan best{0, 0, 0, 1e30, (((M + 127) / 128) * (long)nblocks + cus - 1) / cus * t_small};
    for (int k = 0; k <= 16; ++k) {
        const int big = tiles - k * 32;
        if (big < 0) break;
        const int small = 2 * (tiles - big) + strip * nblocks;
        const int q = big / cus, rem = big % cus; // rounds of big tiles; compute units with one more
        double us = (q + (rem > 0)) * t_big;
        int r = 0;
        while (small) { // rounds of small tiles on the compute units without the extra big one
            const double t = q * t_big + ++r * t_small, after = t - (q + 1) * t_big;
            const long late = after >= 0 ? (long)(after / t_small) : 0; // ... and on the others
            if ((long)(cus - rem) * r + rem * late < small) continue;
            if (t > us) us = t;
            break;
        }
        if (us < best.us) best = {big, small, r, us, best.us_128};
    }
    return best;
}

int launch_gemm_wk_big(hipStream_t st, const rkh_gemm_args& g, rkk::BigTiles plan) {
    const int nblocks = (g.N + 255) / 256, mblocks = g.M / 256 + (g.M % 256 > 128);
    // A workgroup per compute unit takes tile after tile; a K of fewer steps than the look-ahead, where the loads that run ahead
    // would have to pass over a whole tile, gets a workgroup per tile.
    const int cus = compute_units() > 0 ? compute_units() : 256, total = plan.big + plan.small;
    const bool chained = rkh_align_up(g.K, RKH_K_ALIGN) >= 512 && total > cus;
    const dim3 grid(chained ? cus : total), block(512);
    mark(st, "gemm_wk_big_kernel");
#define RK_WKB(W4, EPI)                                                                             \
    do {                                                                                            \
        static std::atomic<bool> opted_in[64] = {};                                                 \
        int dev = 0;                                                                                \
        RKH_CHECK(hipGetDevice(&dev));                                                              \
        if (dev < 0 || dev >= 64) return RKH_ERR_RUNTIME;                                           \
        if (!opted_in[dev].load(std::memory_order_acquire)) {                                       \
            RKH_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_wk_big_kernel<W4, EPI>), \
                                          hipFuncAttributeMaxDynamicSharedMemorySize, WK_LDS_BYTES)); \
            opted_in[dev].store(true, std::memory_order_release);                                   \
        }                                                                                           \
        hipLaunchKernelGGL((gemm_wk_big_kernel<W4, EPI>), grid, block, WK_LDS_BYTES, st,           \
                           g.A, g.W, g.M, g.K, mblocks, nblocks, plan.big, plan.small, chained ? plan.rounds : 0, g);                      \
    } while (0)
    switch (g.epilogue) {
    case RKH_EPI_I32: if (g.w_int4) RK_WKB(true, RKH_EPI_I32); else RK_WKB(false, RKH_EPI_I32); break;
    case RKH_EPI_F16: if (g.w_int4) RK_WKB(true, RKH_EPI_F16); else RK_WKB(false, RKH_EPI_F16); break;
    case RKH_EPI_F32: if (g.w_int4) RK_WKB(true, RKH_EPI_F32); else RK_WKB(false, RKH_EPI_F32); break;
    case RKH_EPI_SWIGLU: if (g.w_int4) RK_WKB(true, RKH_EPI_SWIGLU); else return RKH_ERR_RUNTIME; break;
    default: return RKH_ERR_RUNTIME;
    }
#undef RK_WKB
    RKH_CHECK(hipGetLastError());
    return RKH_OK;
}

// Tiles of 64 or 128 rows x 128 columns (one column block per wave), K not split over workgroups: a few
// hundred rows whose 256-column tiles would leave compute units without one.  The activation rows of a tile
// go through LDS once for the eight waves, so a tile pulls K x (rows + 128) bytes through its compute unit.
template <int TM>
int launch_gemm_wk_narrow(hipStream_t st, const rkh_gemm_args& g) {
    constexpr int TN = 1;
    const int mblocks = (g.M + 32 * TM - 1) / (32 * TM), nblocks = (g.N + 127) / 128;
    const int units = (int)(rkh_align_up(g.K, RKH_K_ALIGN) / WK_PART_K);
    const dim3 grid(mblocks * nblocks), block(512);
    mark(st, TM == 2 ? "gemm_wk_kernel<64 x 128>" : "gemm_wk_kernel<128 x 128>");
#define RK_WKN(W4, EPI, RAW)                                                                        \
    do {                                                                                            \
        static std::atomic<bool> opted_in[64] = {};                                                 \
        int dev = 0;                                                                                \
        RKH_CHECK(hipGetDevice(&dev));                                                              \
        if (dev < 0 || dev >= 64) return RKH_ERR_RUNTIME;                                           \
        if (!opted_in[dev].load(std::memory_order_acquire)) {                                       \
            RKH_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_wk_kernel<TM, W4, EPI, TN, RAW>), \
                                          hipFuncAttributeMaxDynamicSharedMemorySize, WK_LDS_BYTES)); \
            opted_in[dev].store(true, std::memory_order_release);                                   \
        }                                                                                           \
        hipLaunchKernelGGL((gemm_wk_kernel<TM, W4, EPI, TN, RAW>), grid, block, WK_LDS_BYTES, st,       \
                           g.A, g.W, g.M, g.K, mblocks, nblocks, 1, units, g);               \
    } while (0)
    // (int4 weights: the 64-row tiles only -- the 128-row ones measured slower than the other plans everywhere)
#define RK_WKN_W(EPI)                                                                               \
    do {                                                                                            \
        if (!g.w_int4) RK_WKN(false, EPI, false);                                                   \
        else if constexpr (TM == 2) RK_WKN(true, EPI, false);                                            \
        else return RKH_ERR_RUNTIME;                                                                \
    } while (0)
    switch (g.epilogue) {
    case RKH_EPI_I32:
        if (g.A_rows && !g.w_int4) RK_WKN(false, RKH_EPI_I32, true);
        else RK_WKN_W(RKH_EPI_I32);
        break;
    case RKH_EPI_F16: RK_WKN_W(RKH_EPI_F16); break;
    case RKH_EPI_F32: RK_WKN_W(RKH_EPI_F32); break;
    default: return RKH_ERR_RUNTIME;
    }
#undef RK_WKN_W
#undef RK_WKN
    RKH_CHECK(hipGetLastError());
    return RKH_OK;
}

} // namespace

namespace rkk {
// (the tiles owed to the caller are written a few per wave, at most RAW_TILES: K up to 4 N for 64 rows, 2 N for 128; a lane's
// place in its rows is 32 bits)
bool wk_takes_rows(const rkh_gemm_args& g, const void* rows, int tile_rows) {
    const long nb = (g.N + 127) / 128, tiles = tile_rows / 32 * (long)(rkh_align_up(g.K, RKH_K_ALIGN) / 32);
    return !g.w_int4 && g.epilogue == RKH_EPI_I32 && g.K % 16 == 0 && reinterpret_cast<uintptr_t>(rows) % 16 == 0 && g.K <= 1 << 24 &&
           (tiles + nb - 1) / nb <= 8 * RAW_TILES;
}
int launch_gemm_wk_narrow(hipStream_t st, const rkh_gemm_args& g, int tile_rows) {
    return tile_rows == 128 ? ::launch_gemm_wk_narrow<4>(st, g) : ::launch_gemm_wk_narrow<2>(st, g);
}
BigTiles wk_big_tiles(int M, int N, int K, int w_int4) {
    const BigPlan plan = big_plan(M, N, K, w_int4);
    return {plan.big, plan.small, plan.rounds};
}
bool wk_big_applies(int M, int N, int K, int w_int4, BigTiles* tiles) {
    // (as many tiles of 128 x 256 as compute units run in one round: nothing to gain, and other plans may be better still)
    if ((M + 127) / 128 * (long)((N + 255) / 256) <= (compute_units() > 0 ? compute_units() : 256)) return false;
    const BigPlan plan = big_plan(M, N, K, w_int4);
    *tiles = {plan.big, plan.small, plan.rounds};
    return plan.big > 0 && plan.us < plan.us_128;
}
int launch_gemm_wk_big(hipStream_t st, const rkh_gemm_args& g, BigTiles tiles) { return ::launch_gemm_wk_big(st, g, tiles); }
size_t wk_scratch_bytes(long tiles, int bm, int ksplit) { return ::wk_scratch_bytes(tiles, bm, ksplit); }
int launch_gemm_wk(hipStream_t st, const rkh_gemm_args& g, int tile_rows, int ksplit) {
    if (tile_rows == 128) return ::launch_gemm_wk<4>(st, g, ksplit);
    if (tile_rows == 64) return ::launch_gemm_wk<2>(st, g, ksplit);
    return ::launch_gemm_wk<1>(st, g, ksplit);
}
#ifdef RK_DEBUG_TS
void set_ts_gemm(unsigned long long* p) { (void)hipMemcpyToSymbol(HIP_SYMBOL(rk_dbg_ts), &p, sizeof(p)); }
#endif
} // namespace rkk
