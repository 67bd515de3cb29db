// Kernel template of the dequant-fused weight-only GEMM for many activation rows (M > 32), the
// prefill shape.  Included by one translation unit per weight kind (qgemm_mfma_*.hip) so that
// the instantiations compile in parallel.
// Replaces MMHelper::compute* (reference src/utils/matmul_helper.h:565-1705) at large M, where
// the reference switches to AMX (oneDNN) kernels.  MFMA-bound.
//
// A workgroup of 4 wavefronts computes a (4*WN*32 columns) x (WM*32 rows) output tile.  Each
// wave owns WN column tiles and streams their packed codes from global memory straight into
// registers (the same 1-KiB tile layout the M <= 32 kernel uses: a 128-bit load per lane becomes
// MFMA "B" operands after widening), so weights never pass through LDS.  The activation rows are
// shared by the 4 waves: staged through three padded LDS tiles and read back as 128-bit "A"
// operands.  The k loop is a three-stage pipeline (weights two tiles ahead in registers,
// activations four tiles ahead in registers and two in LDS) whose memory instructions are spread
// over the MFMAs of a step; the widening of each operand runs one MFMA group ahead of its use.
// Scale / zero-point / bias / activation / residual are applied in the epilogue.
#pragma once
#include "qgemm_direct_impl.h"
#include "qgemm_mfma_common.h"

namespace xfthip {
namespace {

// MFMA shape: v_mfma_f32_32x32x16_bf16 with the activations as the "A" operand (rows = tokens)
// and the widened weights as "B" (columns = output columns), so a lane's accumulators are
// D[m = 8 (j/4) + 4 h + j%4][n = lane & 31] (h = lane >> 5): consecutive lanes hold consecutive
// output columns and the epilogue stores 64-byte row segments.
//
// KIND: weight kind; WN: 32-column tiles per wave (4 waves per block split the columns);
// WM: 32-row activation tiles per block (shared by the waves through LDS); NEED_SUM: accumulate
// row sums of A for the zero-point term; KTAIL: K is not a whole number of tiles.
template <int KIND>
struct StepTraits;
template <>
struct StepTraits<XFTHIP_W_INT8> {
    // a lane of half h takes the whole 16-byte chunks of k groups h and 2 + h (one 128-bit load each):
    // the k index of an MFMA is only a summation index, so lane half h of micro-step (g, sb) stands for
    // k = 32 g + 16 h + 8 sb .. + 7 in both operands
    static constexpr int KTILE = 64, GROUPS = 2, SUB = 2, WREGS = 4, PACKED_K = 64;
};
template <>
struct StepTraits<XFTHIP_W_UINT4> {
    // 16 bytes per lane per k group, 2 MFMAs.  A step covers half a packed tile (two of its four k groups): with the
    // whole 128-deep tile a step the three activation buffers of a 128-row block take 104 KB of LDS, one workgroup a CU
    static constexpr int KTILE = 64, GROUPS = 2, SUB = 2, WREGS = 4, PACKED_K = 128;
};
template <>
struct StepTraits<XFTHIP_W_NF4> {
    static constexpr int KTILE = 64, GROUPS = 2, SUB = 2, WREGS = 4, PACKED_K = 128;
};
template <>
struct StepTraits<XFTHIP_W_BF16> {
    static constexpr int KTILE = 32, GROUPS = 2, SUB = 1, WREGS = 4, PACKED_K = 32;
};

// DEVROWS: the row count (and, for a group of weights, the weight) comes from device memory (SkinnyParams::rows_dev /
// group); a form of its own, so that the plain kernels carry none of it
template <int KIND, int WN, int WM, bool NEED_SUM, bool KTAIL, bool DEVROWS = false, int WSETS = 3>
__global__ __launch_bounds__(256, 1) void qgemm_mfma_kernel(SkinnyParams p, int nblocks_n, int nblocks_m) {
    using T = StepTraits<KIND>;
    constexpr int KTILE = T::KTILE, GROUPS = T::GROUPS, SUB = T::SUB, WREGS = T::WREGS;
    constexpr int PACKED_K = T::PACKED_K, STEPS_PER_TILE = PACKED_K >= KTILE ? PACKED_K / KTILE : 1; // k of a packed 1-KiB tile; steps that share one
    constexpr int ROWS = 32 * WM;
    constexpr int ROWB = KTILE * 2 + 16; // LDS row pitch in bytes
    constexpr int CHUNKS_PER_ROW = KTILE / 8; // 16-byte chunks
    constexpr int TOTAL_CHUNKS = ROWS * CHUNKS_PER_ROW;
    constexpr int ALOADS = TOTAL_CHUNKS / 256;
    static_assert(TOTAL_CHUNKS % 256 == 0, "activation tile must split evenly over the block");
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int h = lane >> 5, nl = lane & 31;
    int nb, m0;
    if (!take_block<ROWS, PACKED_K, DEVROWS>(p, nblocks_n, nblocks_m, lane, nb, m0)) return;
    const int n32_0 = (nb * 4 + wave) * WN; // first 32-column tile of this wave
    uint2 *lut = nullptr;
    unsigned char *abuf_base = lds;
    if constexpr (KIND == XFTHIP_W_NF4) {
        lut = (uint2 *)lds;
        abuf_base = lds + 2048;
        {
            const int i = threadIdx.x;
            const float c0 = c_nf4_big[i & 15], c1 = c_nf4_big[i >> 4];
            const uint32_t h0 = f32_to_bf16_ref(c0), h1 = f32_to_bf16_ref(c1);
            const uint32_t l0 = f32_to_bf16_ref(c0 - bf16_to_f32((uint16_t)h0));
            const uint32_t l1 = f32_to_bf16_ref(c1 - bf16_to_f32((uint16_t)h1));
            lut[i] = make_uint2(h0 | (h1 << 16), l0 | (l1 << 16));
        }
    }

    f32x16 acc[WN][WM];
    f32x16 accS[WM];
#pragma unroll
    for (int t = 0; t < WN; ++t)
#pragma unroll
        for (int m = 0; m < WM; ++m)
#pragma unroll
            for (int j = 0; j < 16; ++j) acc[t][m][j] = 0.0f;
#pragma unroll
    for (int m = 0; m < WM; ++m)
#pragma unroll
        for (int j = 0; j < 16; ++j) accS[m][j] = 0.0f;

    // weight source of this lane: 16-column packed tile (2 per 32-column MFMA tile), chunk of
    // its column inside the tile, and which 8-byte half (INT8) / dword pair (4-bit) it uses
    const XFT_GLOBAL uint8_t *wbase[WN];
#pragma unroll
    for (int t = 0; t < WN; ++t) {
        int nt = (n32_0 + t) * 2 + (nl >> 4);
        nt = nt < p.NTILES ? nt : p.NTILES - 1;
        wbase[t] = global_bytes(p.packed) + (size_t)nt * p.KT * 1024 + (nl & 15) * 16;
    }
    constexpr int ROW_STEP = 256 / CHUNKS_PER_ROW;
    const int a_kc = threadIdx.x % CHUNKS_PER_ROW;
    const int a_row0 = threadIdx.x / CHUNKS_PER_ROW;
    uint32_t a_off[ALOADS];
#pragma unroll
    for (int i = 0; i < ALOADS; ++i) {
        int row = m0 + a_row0 + i * ROW_STEP;
        row = row < p.M ? row : p.M - 1;
        if constexpr (DEVROWS) row = p.a_rows ? p.a_rows[row] : row;
        a_off[i] = (uint32_t)row * (uint32_t)p.lda + a_kc * 8;
    }

    const u32x4 zero4 = {0u, 0u, 0u, 0u};
    // Three-stage pipeline over k tiles.  At the start of step k: LDS buffers k % 3 and (k + 1) % 3 hold the
    // activation tiles k and k + 1 (published by earlier barriers), the weight registers of sets k % WSETS
    // .. (k + WSETS - 2) % WSETS hold or await tiles k .. k + WSETS - 2, the activation registers await tile k + 2,
    // and the first MFMA operands of tile k are already in registers.  Step k sends the loads of weight
    // tile k + WSETS - 1 and activation tile k + 4, moves activation tile k + 2 from registers into LDS buffer
    // (k + 2) % 3 (last read two steps ago), computes tile k while reading each next operand set a
    // micro-step ahead (the last one from tile k + 1's buffer), and ends in the barrier that publishes
    // buffer (k + 2) % 3.  Every wait is for loads at least one full step old, and the MFMAs after a
    // barrier never wait for an LDS read.
    constexpr int MICRO = GROUPS * SUB;
    // weight register sets: tile j in set j % WSETS, loaded WSETS - 1 steps ahead.  Three for the large tiles (MFMA
    // bound; the registers are the accumulators'); six for the 32- and 64-row tiles, whose launches are bound by
    // the weights' trip from HBM - with two tiles in flight a step of such a workgroup waited most of a round trip
    static_assert(WSETS % 3 == 0, "the activation side of the pipeline walks three buffers");
    constexpr int WD = WSETS - 1;
    uint32_t wreg[WSETS][GROUPS][WN][WREGS];
    u32x4 areg[3][ALOADS];
    const int kt_n = (p.K + KTILE - 1) / KTILE;

    // weight codes of k group gq of tile kt_ into register set buf
    auto load_w_part = [&](int buf, int kt_, int gq) {
        const int kt = kt_ < kt_n ? kt_ : kt_n - 1; // past the end: a valid tile, never used
#pragma unroll
        for (int t = 0; t < WN; ++t) {
            if constexpr (KIND == XFTHIP_W_INT8) {
                const u32x4 v = *(const XFT_GLOBAL u32x4 *)(wbase[t] + (size_t)kt * 1024 + (2 * gq + h) * 256);
                wreg[buf][gq][t][0] = v[0]; wreg[buf][gq][t][1] = v[1]; wreg[buf][gq][t][2] = v[2]; wreg[buf][gq][t][3] = v[3];
            } else if constexpr (KIND == XFTHIP_W_BF16) {
                // chunk g = 2 s + h holds k = 8 g .. 8 g + 7
                const u32x4 v = *(const XFT_GLOBAL u32x4 *)(wbase[t] + (size_t)kt * 1024 + (2 * gq + h) * 256);
                wreg[buf][gq][t][0] = v[0]; wreg[buf][gq][t][1] = v[1]; wreg[buf][gq][t][2] = v[2]; wreg[buf][gq][t][3] = v[3];
            } else {
                const u32x4 v = *(const XFT_GLOBAL u32x4 *)(wbase[t] + (size_t)(kt / STEPS_PER_TILE) * 1024 + ((kt % STEPS_PER_TILE) * GROUPS + gq) * 256);
                wreg[buf][gq][t][0] = v[0]; wreg[buf][gq][t][1] = v[1]; wreg[buf][gq][t][2] = v[2]; wreg[buf][gq][t][3] = v[3];
            }
        }
    };
    auto load_w = [&](int buf, int kt_) {
#pragma unroll
        for (int gq = 0; gq < GROUPS; ++gq) load_w_part(buf, kt_, gq);
    };
    // 16-byte chunk i of this thread's share of activation tile kt_ into register set `set`
    auto load_a_part = [&](int set, int kt_, int i) {
        const int kt = kt_ < kt_n ? kt_ : kt_n - 1;
        if constexpr (KTAIL) {
            const int k = kt * KTILE + a_kc * 8;
            const bool v = k < p.K;
            const u32x4 a = *(const u32x4 *)(p.A + a_off[i] + (v ? (size_t)kt * KTILE : (size_t)0) - (v ? 0 : a_kc * 8));
            areg[set][i] = v ? a : zero4;
        } else {
            areg[set][i] = *(const u32x4 *)(p.A + a_off[i] + (size_t)kt * KTILE);
        }
    };
    auto load_a = [&](int set, int kt_) {
#pragma unroll
        for (int i = 0; i < ALOADS; ++i) load_a_part(set, kt_, i);
    };
    // NEED_SUM: the row sums of A (zero-point term) are gathered where the rows are staged: the thread that moves a
    // 16-byte chunk into LDS adds its 8 values to a partial of its own; the partials of a row's chunks are joined after
    // the k loop.  (They used to come from one more MFMA a row tile and micro-step against a tile of ones: as many
    // MFMAs again as the product itself with one column tile a wave, and 16 WM accumulator registers.)
    float rs_part[ALOADS];
#pragma unroll
    for (int i = 0; i < ALOADS; ++i) rs_part[i] = 0.0f;
    auto store_a_part = [&](int set, int buf, int i, bool real_tile) {
        unsigned char *dst = abuf_base + buf * (ROWS * ROWB);
        *(u32x4 *)(dst + (a_row0 + i * ROW_STEP) * ROWB + a_kc * 16) = areg[set][i];
        if constexpr (NEED_SUM) {
            if (real_tile) { // (uniform: tiles past the end of K are copies of the last one)
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const uint32_t u = areg[set][i][w];
                    rs_part[i] += u2f(u << 16) + u2f(u & 0xFFFF0000u);
                }
            }
        }
    };
    auto store_a = [&](int set, int buf, bool real_tile) {
#pragma unroll
        for (int i = 0; i < ALOADS; ++i) store_a_part(set, buf, i, real_tile);
    };
    // k offset (elements) of micro-step ms inside a tile: lane (row/col, h) holds k = koff .. koff + 7
    auto koff_of = [&](int ms) {
        const int gq = ms / SUB, sb = ms % SUB;
        return KIND == XFTHIP_W_INT8 ? 32 * gq + 16 * h + 8 * sb : KIND == XFTHIP_W_BF16 ? 16 * gq + 8 * h : 32 * gq + 16 * sb + 8 * h;
    };
    MFrag afr[2][WM];
    auto read_frags = [&](int slot, int ab, int ms) {
        const unsigned char *src = abuf_base + ab * (ROWS * ROWB) + nl * ROWB + koff_of(ms) * 2;
#pragma unroll
        for (int m = 0; m < WM; ++m) afr[slot][m].q = *(const u32x4 *)(src + m * 32 * ROWB);
    };
    // one MFMA k step = 16 k.  Operands of micro-step ms sit in afr[ms & 1]; the next set (of the
    // next tile's buffer after the last micro-step) is read while this one's MFMAs run.
    // Besides the MFMAs of tile kt (weight set w_cur, LDS buffer lds_cur), a step sends the loads of weight
    // tile kt + WD (into set w_load) and activation tile kt + 4 (into register set a_load) and moves
    // activation tile kt + 2 (register set a_stage, loaded two steps ago) into LDS buffer
    // a_stage: one slice of each per micro-step, so that no wave ever queues a burst of memory
    // instructions in front of its MFMAs (a wave issues in order; 4 waves sending 12 loads each right
    // after a barrier kept the MFMA pipes waiting for the address path).
    constexpr int A_EVERY = MICRO % ALOADS == 0 ? MICRO / ALOADS : 1;
    static_assert(ALOADS <= MICRO, "at most an activation slice a micro-step");
    // UINT4: mask and exponent of a pair of codes in a scalar and a vector register of their own, so that they are one instruction (v_and_or_b32 takes no literal)
    uint32_t nib_mask = 0x000F000Fu, nib_bits = 0x43004300u;
    if constexpr (KIND == XFTHIP_W_UINT4) asm("" : "+s"(nib_mask), "+v"(nib_bits));
    // widened MFMA operands of (weight set wb, micro-step ms, column tile t)
    auto widen = [&](int wb, int ms, int t, MFrag &whi, MFrag &wlo) {
        const int gq = ms / SUB, sb = ms % SUB;
        if constexpr (KIND == XFTHIP_W_INT8) {
            const uint32_t x = wreg[wb][gq][t][2 * sb], y = wreg[wb][gq][t][2 * sb + 1];
            whi.u[0] = pack_hi16_m((float)(int)(int8_t)(x), (float)(int)(int8_t)(x >> 8));
            whi.u[1] = pack_hi16_m((float)(int)(int8_t)(x >> 16), (float)((int)x >> 24));
            whi.u[2] = pack_hi16_m((float)(int)(int8_t)(y), (float)(int)(int8_t)(y >> 8));
            whi.u[3] = pack_hi16_m((float)(int)(int8_t)(y >> 16), (float)((int)y >> 24));
        } else if constexpr (KIND == XFTHIP_W_BF16) {
            whi.u[0] = wreg[wb][gq][t][0]; whi.u[1] = wreg[wb][gq][t][1];
            whi.u[2] = wreg[wb][gq][t][2]; whi.u[3] = wreg[wb][gq][t][3];
        } else {
            // codes 16 sb + 8 h .. + 8 of the lane's 32-code chunk = dword 2 sb + h
            const uint32_t x0 = wreg[wb][gq][t][2 * sb], x1 = wreg[wb][gq][t][2 * sb + 1];
            const uint32_t x = h ? x1 : x0;
            if constexpr (KIND == XFTHIP_W_UINT4) {
                whi.u[0] = (x & nib_mask) | nib_bits;
                whi.u[1] = ((x >> 4) & nib_mask) | nib_bits;
                whi.u[2] = ((x >> 8) & nib_mask) | nib_bits;
                whi.u[3] = ((x >> 12) & nib_mask) | nib_bits;
            } else {
                const uint2 e0 = lut[x & 0xFF], e1 = lut[(x >> 8) & 0xFF], e2 = lut[(x >> 16) & 0xFF], e3 = lut[x >> 24];
                whi.u[0] = e0.x; whi.u[1] = e1.x; whi.u[2] = e2.x; whi.u[3] = e3.x;
                wlo.u[0] = e0.y; wlo.u[1] = e1.y; wlo.u[2] = e2.y; wlo.u[3] = e3.y;
            }
        }
    };
    // The operands of slot (ms, t) are widened while the MFMAs of the slot before run: wcur_* enter
    // a step holding slot (0, 0) of its tile and leave it holding slot (0, 0) of the next tile.
    MFrag wcur_hi, wcur_lo;
    // the explicit interleave below pays for the BF16 kind (no widening work to hide: +5 %) and costs
    // the INT8 kind 6 % on 128 x 128 tiles, where the compiler's own order is better
    constexpr bool SGB = KIND == XFTHIP_W_BF16;
    // VALU instructions one widening takes (a hint for the instruction interleave below)
    constexpr int VW = KIND == XFTHIP_W_INT8 ? 12 : KIND == XFTHIP_W_UINT4 ? 9 : KIND == XFTHIP_W_NF4 ? 6 : 0;
    constexpr int VPER = (VW + WM - 1) / WM;
    // w_cur / w_next / w_load: weight register sets of tiles kt_cur, kt_cur + 1 and kt_cur + WD (the one this step loads).
    // lds_cur / lds_next: LDS tiles of activation tiles kt_cur and kt_cur + 1; a_load: the register set tile kt_cur + 4 is loaded
    // into; a_stage: the register set (and LDS tile of the same number) tile kt_cur + 2 moves from (to)
    auto compute = [&](int w_cur, int w_next, int w_load, int a_load, int a_stage, int kt_cur, int lds_cur, int lds_next) {
#pragma unroll
        for (int ms = 0; ms < MICRO; ++ms) {
            const int gq = ms / SUB, sb = ms % SUB;
            if (sb == 0) load_w_part(w_load, kt_cur + WD, gq);
            if (ms % A_EVERY == 0 && ms / A_EVERY < ALOADS) {
                load_a_part(a_load, kt_cur + 4, ms / A_EVERY);
                store_a_part(a_stage, a_stage, ms / A_EVERY, kt_cur + 2 < kt_n);
            }
            if (ms + 1 < MICRO)
                read_frags((ms + 1) & 1, lds_cur, ms + 1);
            else
                read_frags((ms + 1) & 1, lds_next, 0);
            const MFrag *a = afr[ms & 1];
#pragma unroll
            for (int t = 0; t < WN; ++t) {
                MFrag nhi, nlo;
                if (t + 1 < WN)
                    widen(w_cur, ms, t + 1, nhi, nlo);
                else if (ms + 1 < MICRO)
                    widen(w_cur, ms + 1, 0, nhi, nlo);
                else
                    widen(w_next, 0, 0, nhi, nlo); // the next tile's set: loaded in an earlier step
#pragma unroll
                for (int m = 0; m < WM; ++m) {
                    if constexpr (KIND == XFTHIP_W_NF4)
                        acc[t][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[m].v, wcur_lo.v, acc[t][m], 0, 0, 0);
                    acc[t][m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[m].v, wcur_hi.v, acc[t][m], 0, 0, 0);
                }
                wcur_hi = nhi;
                if constexpr (KIND == XFTHIP_W_NF4) wcur_lo = nlo;
                if constexpr (SGB) {
                    // order of the slot's instructions: its memory instructions first, then one MFMA at a
                    // time with a share of the widening and (first column tile) one LDS read behind it
                    if (t == 0) {
                        if (sb == 0) {
#pragma unroll
                            for (int tt = 0; tt < WN; ++tt) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                        }
                        if (ms % A_EVERY == 0) {
                            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                            __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);
                        }
                    }
#pragma unroll
                    for (int m = 0; m < WM; ++m) {
                        __builtin_amdgcn_sched_group_barrier(0x008, KIND == XFTHIP_W_NF4 ? 2 : 1, 0);
                        if (t == 0) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                        if (VPER > 0) __builtin_amdgcn_sched_group_barrier(0x002, VPER, 0);
                    }
                }
            }
        }
    };

#define XFT_FENCE() __builtin_amdgcn_sched_barrier(0)
    int kt = 0;
    // prologue: tiles 0 and 1 in LDS, weight tiles 0 and 1 and activation tiles 2 and 3 under way
    load_w(0, 0);
    load_a(0, 0);
    load_w(1, 1);
    load_a(1, 1);
    load_a(2, 2);
#pragma unroll
    for (int i = 2; i < WD; ++i) load_w(i, i);
    XFT_FENCE();
    store_a(0, 0, true);
    XFT_FENCE();
    load_a(0, 3);
    XFT_FENCE();
    store_a(1, 1, kt_n > 1);
    __syncthreads();
    read_frags(0, 0, 0);
    widen(0, 0, 0, wcur_hi, wcur_lo);
    // step k with s = k % 3 (static): tile j lives in weight set, activation register set and LDS buffer j % 3
#define XFT_STEP(s)                                        \
    {                                                      \
        compute((s), ((s) + 1) % WSETS, ((s) + WD) % WSETS, ((s) + 1) % 3, ((s) + 2) % 3, kt, (s) % 3, ((s) + 1) % 3); \
        XFT_FENCE();                                       \
        __syncthreads();                                   \
        ++kt;                                              \
    }
    if constexpr (WSETS == 6) {
        while (kt + 6 <= kt_n) {
            XFT_STEP(0) XFT_STEP(1) XFT_STEP(2) XFT_STEP(3) XFT_STEP(4) XFT_STEP(5)
        }
        if (kt < kt_n) XFT_STEP(0)
        if (kt < kt_n) XFT_STEP(1)
        if (kt < kt_n) XFT_STEP(2)
        if (kt < kt_n) XFT_STEP(3)
        if (kt < kt_n) XFT_STEP(4)
    } else {
        while (kt + 3 <= kt_n) {
            XFT_STEP(0) XFT_STEP(1) XFT_STEP(2)
        }
        if (kt < kt_n) XFT_STEP(0)
        if (kt < kt_n) XFT_STEP(1)
    }
#undef XFT_STEP
#undef XFT_FENCE

    // ---- epilogue: lane holds C[m0 + 32 mt + 8 (j/4) + 4 h + j%4][32 (n32_0 + t) + nl] ----
    // A lane owns 16 rows of ONE column.  Finishing and storing every element from the accumulator
    // registers costs a 64-bit index, bounds tests and a type conversion in 128 unrolled copies a
    // lane, which made the epilogue of a 2048 x 4096 result take 23 us (the k loop of K = 4096: 75).
    // Instead each wave drops one 32-row block of scaled results at a time, as fp32, into an LDS
    // patch of its own (one ds_write with a constant offset per element), then walks the patch in
    // 8-column chunks, consecutive lanes along a row: residual, conversion and 16-byte stores run
    // in that short loop.
    constexpr int OPITCH = 32 * WN * 4 + 32; // patch row pitch in bytes
    __syncthreads(); // every wave is past its last read of the activation tiles
    unsigned char *obuf = abuf_base + wave * (32 * OPITCH);
    if constexpr (NEED_SUM) {
        // join the partial sums of a row's chunks (adjacent lanes), hand them over through LDS behind the patches, and
        // give every lane the sums of the 16 rows it holds results of
        float *rowsum = (float *)(abuf_base + 4 * 32 * OPITCH);
#pragma unroll
        for (int i = 0; i < ALOADS; ++i) {
            float v = rs_part[i];
#pragma unroll
            for (int off = 1; off < CHUNKS_PER_ROW; off <<= 1) v += __shfl_xor(v, off, 64);
            if (a_kc == 0) rowsum[a_row0 + i * ROW_STEP] = v;
        }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < WM; ++m)
#pragma unroll
            for (int j = 0; j < 16; ++j) accS[m][j] = rowsum[32 * m + 8 * (j >> 2) + 4 * h + (j & 3)];
    }
    const FlushRows to = flush_target(p, obuf, OPITCH, lane);
    auto put_at = [&](float *base, int t_cols, int j, float x) { base[(8 * (j >> 2) + (j & 3)) * (OPITCH / 4) + t_cols] = x; };
    auto run_epilogue = [&](auto epi_tag) {
        constexpr int EPI = decltype(epi_tag)::value;
        float s[WN], z[WN], bv[WN];
#pragma unroll
        for (int t = 0; t < WN; ++t) {
            const int np = (n32_0 + t) * 32 + nl;
            s[t] = 1.0f, z[t] = 0.0f, bv[t] = 0.0f;
            if constexpr (KIND != XFTHIP_W_BF16) s[t] = p.scale[np < p.NTILES * 16 ? np : 0];
            if constexpr (KIND == XFTHIP_W_UINT4 || (KIND == XFTHIP_W_INT8 && NEED_SUM)) z[t] = p.zero ? p.zero[np < p.NTILES * 16 ? np : 0] : 0.0f;
            if constexpr (EPI == XFTHIP_EPI_BIAS || EPI == XFTHIP_EPI_RESIDENTIAL || EPI == XFTHIP_EPI_RESEXT) bv[t] = (p.bias && np < p.N) ? p.bias[np] : 0.0f;
        }
        float *put_base = (float *)(obuf + 4 * h * OPITCH) + nl;
#pragma unroll
        for (int m = 0; m < WM; ++m) {
#pragma unroll
            for (int t = 0; t < WN; ++t) {
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    float x = acc[t][m][j];
                    if constexpr (KIND == XFTHIP_W_UINT4) {
                        x = fmaf(s[t], x - 128.0f * accS[m][j], z[t] * accS[m][j]);
                    } else if constexpr (KIND == XFTHIP_W_INT8) {
                        x = s[t] * x;
                        if constexpr (NEED_SUM) x = fmaf(z[t], accS[m][j], x);
                    } else if constexpr (KIND == XFTHIP_W_NF4) {
                        x = s[t] * x;
                    }
                    if constexpr (EPI == XFTHIP_EPI_BIAS || EPI == XFTHIP_EPI_RESIDENTIAL || EPI == XFTHIP_EPI_RESEXT) x += bv[t];
                    if constexpr (EPI == XFTHIP_EPI_SILU) x = silu_big(x);
                    if constexpr (EPI == XFTHIP_EPI_GELU) {
                        const float e = fast_exp(1.702f * x);
                        x = e / (e + 1.0f) * x;
                    }
                    put_at(put_base, 32 * t, j, x); // the residual operand joins in flush_rows()
                }
            }
            flush_rows<EPI>(to, p, m0 + 32 * m, n32_0 * 32, 32 * WN, p.N);
        }
    };
    if (p.gateup) {
        // packed columns alternate 16 gate / 16 up: lanes nl < 16 hold gate, nl >= 16 the matching up
        float s[WN], z[WN], bv[WN];
#pragma unroll
        for (int t = 0; t < WN; ++t) {
            const int np = (n32_0 + t) * 32 + nl, col = (n32_0 + t) * 16 + (nl & 15);
            s[t] = 1.0f, z[t] = 0.0f;
            bv[t] = p.bias && col < p.N / 2 ? p.bias[(nl < 16 ? 0 : p.N / 2) + col] : 0.0f;
            if constexpr (KIND != XFTHIP_W_BF16) s[t] = p.scale[np < p.NTILES * 16 ? np : 0];
            if constexpr (KIND == XFTHIP_W_UINT4 || (KIND == XFTHIP_W_INT8 && NEED_SUM)) z[t] = p.zero ? p.zero[np < p.NTILES * 16 ? np : 0] : 0.0f;
        }
        // gate lanes write output column 16 t + nl of the strip; the up lanes' copies of the
        // product land in the unused columns behind the strip, which flush_rows() never reads
        float *put_base = (float *)(obuf + 4 * h * OPITCH) + (nl < 16 ? nl : 16 * WN + (nl - 16));
#pragma unroll
        for (int m = 0; m < WM; ++m) {
#pragma unroll
            for (int t = 0; t < WN; ++t) {
#pragma unroll
                for (int j = 0; j < 16; ++j) {
                    float x = acc[t][m][j];
                    if constexpr (KIND == XFTHIP_W_UINT4) {
                        x = fmaf(s[t], x - 128.0f * accS[m][j], z[t] * accS[m][j]);
                    } else if constexpr (KIND == XFTHIP_W_INT8) {
                        x = s[t] * x;
                        if constexpr (NEED_SUM) x = fmaf(z[t], accS[m][j], x);
                    } else if constexpr (KIND == XFTHIP_W_NF4) {
                        x = s[t] * x;
                    }
                    x += bv[t];
                    const float other = __shfl_xor(x, 16, 64); // gate <-> up partner
                    put_at(put_base, 16 * t, j, p.gateup == 2 ? clamped_glu(x, other, p.glu_limit, p.glu_alpha) : other * silu_big(x));
                }
            }
            flush_rows<XFTHIP_EPI_NONE>(to, p, m0 + 32 * m, n32_0 * 16, 16 * WN, p.N / 2);
        }
        return;
    }
    switch (p.epi) {
        case XFTHIP_EPI_BIAS: run_epilogue(std::integral_constant<int, XFTHIP_EPI_BIAS> {}); break;
        case XFTHIP_EPI_SILU: run_epilogue(std::integral_constant<int, XFTHIP_EPI_SILU> {}); break;
        case XFTHIP_EPI_GELU: run_epilogue(std::integral_constant<int, XFTHIP_EPI_GELU> {}); break;
        case XFTHIP_EPI_RESMUL: run_epilogue(std::integral_constant<int, XFTHIP_EPI_RESMUL> {}); break;
        case XFTHIP_EPI_RESIDENTIAL: run_epilogue(std::integral_constant<int, XFTHIP_EPI_RESIDENTIAL> {}); break;
        case XFTHIP_EPI_RESEXT: run_epilogue(std::integral_constant<int, XFTHIP_EPI_RESEXT> {}); break;
        default: run_epilogue(std::integral_constant<int, XFTHIP_EPI_NONE> {}); break;
    }
}

template <int KIND, int WN, int WM, bool NEED_SUM, bool KTAIL, bool DEVROWS = false>
static int launch_big2(const SkinnyParams &p, hipStream_t stream) {
    // six weight tiles in flight for the 32- and 64-row tiles (see the kernel), three for the others
    constexpr int WSETS = WN == 1 && WM <= 2 ? 6 : 3, ROWS = 32 * WM, ROWB = StepTraits<KIND>::KTILE * 2 + 16;
    BlockGrid g;
    if (int rc = block_grid<DEVROWS>(p, ROWS, 8 * WN, g)) return rc;
    // the three activation buffers, reused after the k loop by the four waves' output patches
    // (the row sums of the zero-point term sit behind the patches)
    const size_t pipe = 3 * ROWS * ROWB, patches = 4 * 32 * (32 * WN * 4 + 32) + (NEED_SUM ? ROWS * sizeof(float) : 0);
    const size_t smem = (pipe > patches ? pipe : patches) + (KIND == XFTHIP_W_NF4 ? 2048 : 0);
    if (smem > 64 * 1024) {
        // more dynamic LDS than the default limit: raise it once per instantiation
        static const hipError_t attr = hipFuncSetAttribute((const void *)qgemm_mfma_kernel<KIND, WN, WM, NEED_SUM, KTAIL, DEVROWS, WSETS>,
                hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        XFT_CHECK_HIP(attr);
    }
    SkinnyParams q = p;
    q.band = g.band;
    hipLaunchKernelGGL((qgemm_mfma_kernel<KIND, WN, WM, NEED_SUM, KTAIL, DEVROWS, WSETS>), dim3(g.blocks), dim3(256), smem, stream, q, g.nblocks_n, g.nblocks_m);
    XFT_CHECK_HIP(hipGetLastError());
    return 0;
}

template <int KIND, int WN, int WM, bool NEED_SUM>
static int launch_big(const SkinnyParams &p, hipStream_t stream) {
    if constexpr (WM >= 3) {
        // 96 and 128 rows: the activations straight into LDS, two workgroups a CU, or (at most a block a CU) two K groups a workgroup.  Staged through registers
        // only 128-row tiles, for a ragged K or more than 4 GB of activations.
        if (p.rows_dev) return launch_direct<KIND, 2 * WN, 2 * WM, NEED_SUM, true, 1>(p, stream); // (taken for whole k steps only)
        if constexpr (WM == 4)
            if (p.direct && p.kgroups == 2) return launch_direct<KIND, 2 * WN, 2 * WM, NEED_SUM, false, 2>(p, stream);
        if (p.direct) return launch_direct<KIND, 2 * WN, 2 * WM, NEED_SUM, false, 1>(p, stream);
        if constexpr (WM == 4) {
            if constexpr (WN == 2 || KIND == XFTHIP_W_BF16)
                if (p.K % StepTraits<KIND>::KTILE == 0) return launch_big2<KIND, WN, WM, NEED_SUM, false>(p, stream);
            if constexpr (WN == 2) return launch_big2<KIND, WN, WM, NEED_SUM, true>(p, stream);
        }
        set_error("qgemm_mfma: no tile of %d x %d for this K", 32 * WM, 128 * WN);
        return 2;
    } else {
        const bool ragged = p.K % StepTraits<KIND>::KTILE != 0;
        if (p.rows_dev) return ragged ? launch_big2<KIND, WN, WM, NEED_SUM, true, true>(p, stream) : launch_big2<KIND, WN, WM, NEED_SUM, false, true>(p, stream);
        return ragged ? launch_big2<KIND, WN, WM, NEED_SUM, true>(p, stream) : launch_big2<KIND, WN, WM, NEED_SUM, false>(p, stream);
    }
}

template <int KIND, bool NEED_SUM>
static int dispatch_big_tile(const SkinnyParams &p, hipStream_t stream) {
    switch (p.tile) { // (choose_tile; 5 with activations straight into LDS only)
        case 1:
            if constexpr (KIND != XFTHIP_W_BF16) return launch_big<KIND, 1, 1, NEED_SUM>(p, stream);
            break;
        case 3: return launch_big<KIND, 1, 4, NEED_SUM>(p, stream);
        case 4: return launch_big<KIND, 2, 4, NEED_SUM>(p, stream);
        case 5: return launch_big<KIND, 2, 3, NEED_SUM>(p, stream);
        default: break;
    }
    return launch_big<KIND, 1, 2, NEED_SUM>(p, stream);
}

} // namespace
} // namespace xfthip
