// Kernel of the dequant-fused weight-only GEMM for many activation rows whose activation tiles go from global memory straight into LDS: the 128 x 256,
// 96 x 256 and 128 x 128 block tiles of qgemm_mfma.hip (the smaller tiles and the forms for a ragged K are qgemm_mfma_impl.h's, which includes this file).
// Replaces MMHelper::compute* (reference src/utils/matmul_helper.h:565-1705) at large M.
//
// A workgroup of 4 wavefronts computes 16 RT rows x 64 CT columns; each wave owns CT packed tiles of 16 columns and all rows.  The weights are the MFMA's first
// operand (result rows = output columns), straight from the packed tiles in global memory and widened in registers, the activation rows its second (result
// columns = tokens), read from LDS: a lane's accumulators are 4 neighbouring output columns of one token.
//
// What bounds it is the card's power: on random data the same loop on zeros runs 1.45 times as fast (2048 x 16384 x 16384 INT8 573 us against 835, in the form
// before), at the same waits.  v_mfma_f32_16x16x32_bf16 does a product in less energy than v_mfma_f32_32x32x16_bf16, whose accumulators are read and written
// twice as often: 1.83 against 1.64 PFLOP/s in a loop of MFMAs and operand reads alone, 2.09 against 1.80 in MFMAs alone (2.45 either on zeros).  2048 x 16384,
// K = 4096 / 16384, against that form: INT8 230 / 825 -> 218 / 775 us (1.42 PFLOP/s), UINT4 233 / 788 -> 210 / 710 (1.55), BF16 239 / 906 -> 212 / 866 (1.27);
// 2011 x 11008 x 4096 INT8 155 -> 148, a Mixtral-8x7B layer of 256 tokens 356 -> 333.  What is left beside the products are the bytes they come from: at a step of
// 4 KB a wave the weights' way from L2 is a fifth of the time (INT8, left out: 835 -> 659), the activations' 8 %, the barriers nothing; their way from memory is hidden: 2048 x 11008 x 4096 over
// one weight / eight in turn INT8 153.5 / 155.5 us, UINT4 143.8 / 144.0, BF16 153 / 158.  (Behind an idle device the first 24 launches take 188, 180 and 186, the next 96 166, 158 and 166.)
// Counters of these launches, each by itself: INT8 305,000 clocks at 1.94 GHz, matrix units busy 58 % of them, vector ALUs 42 % (the issue of MFMAs among it), LDS ports 16 %, waves waiting 14 % of their
// time in counted waits; UINT4 329,000 clocks at 2.17 GHz, 54 %, 36 %, 15 %, 13 %.
#pragma once
#include "qgemm_mfma_common.h"

namespace xfthip {
namespace {

// KSTEP: k a step; NBUF: activation tiles in LDS; SETS: weight tiles in registers, three (BF16, 32 registers each: two, reloaded behind the products that read them) but
// for 128 x 128 blocks of four waves, which have room for twice as many and wait for them: 100 x 4096 x 14336, blocks alone on their CUs, INT8 98 -> 89 us, BF16 133 -> 117
// (with two K groups, 96 x 256 and the 4-bit kinds the same or 1 to 3 % slower).
template <int KIND, int CT, int KG>
struct DirectTraits { // 4-bit kinds: a lane holds 32 neighbouring codes, one MFMA takes 8 of each lane group's, so that a step is a whole packed tile of 128 k
    static constexpr int KSTEP = 128, NBUF = 2, SETS = 2;
};
template <int CT, int KG>
struct DirectTraits<XFTHIP_W_INT8, CT, KG> {
    static constexpr int KSTEP = 64, NBUF = 4, SETS = CT == 2 && KG == 1 ? 6 : 3;
};
template <int CT, int KG>
struct DirectTraits<XFTHIP_W_BF16, CT, KG> {
    static constexpr int KSTEP = 64, NBUF = 4, SETS = CT == 2 && KG == 1 ? 4 : 2;
};

// Slot of 16-byte chunk c of LDS row r is c ^ direct_swizzle(r).  A row is 128 or 256 bytes; an operand read is rows 0 .. 15 of a tile, 16 lanes a chunk index,
// the indices of the four lane groups 1, 2 or 4 apart.  Its lanes are served 16 at a time, not always neighbours: 0 .. 3 and 12 .. 15 of one group go with 4 .. 11 of
// the next.  So rows of the two kinds differ in a bit of the slot that the chunk index never touches: no bank conflicts whichever lanes go together.
template <int KSTEP>
__device__ inline int direct_swizzle(int r) {
    if constexpr (KSTEP == 128) return (r & 15) ^ ((r & 4) << 1);
    const int x = (r >> 1) & 7;
    return x ^ ((x & 2) << 1);
}

// an address that is the same in every lane, said so: for a scalar register pair
__device__ inline uint64_t uniform_address(const void *q) {
    const uint64_t bits = (uint64_t)(uintptr_t)q;
    return ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(bits >> 32)) << 32) | (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)bits);
}

// KIND: weight kind; CT: 16-column tiles a wave; RT: 16-row tiles; NEED_SUM: row sums of A for the zero-point term; DEVROWS: row counts (and, for a group of
// weights, the weight) from device memory; KG = 2: two K groups of four waves, each with tiles and a pipeline of its own, for launches of at most a block a CU
// (a SIMD has two waves to issue from, as with two blocks a CU); the second hands its sums to the first through LDS.
template <int KIND, int CT, int RT, bool NEED_SUM, bool DEVROWS, int KG>
__global__ __launch_bounds__(256 * KG, KG == 1 ? 2 : 1) void qgemm_direct_kernel(SkinnyParams p, int nblocks_n, int nblocks_m) {
    using T = DirectTraits<KIND, CT, KG>;
    constexpr int KSTEP = T::KSTEP, NBUF = T::NBUF, WSETS = T::SETS, MICRO = KSTEP / 32;
    constexpr int ROWS = 16 * RT, ROWB = KSTEP * 2, TILEB = ROWS * ROWB, CPR = KSTEP / 8; // bytes of an LDS row and tile, chunks a row
    constexpr int ALOADS = TILEB / 4096;                                                  // requests of 1 KiB a wave and tile
    constexpr bool FOUR = KIND == XFTHIP_W_UINT4 || KIND == XFTHIP_W_NF4, BF16 = KIND == XFTHIP_W_BF16, NF4 = KIND == XFTHIP_W_NF4;
    constexpr int PACKED_K = FOUR ? 128 : BF16 ? 32 : 64, WPARTS = BF16 ? MICRO : 1; // 16-byte weight loads a lane, tile and step
    static_assert(TILEB % 4096 == 0 && (CT == 2 || CT == 4) && (!NEED_SUM || RT == 6 || RT == 8), "tile");
    extern __shared__ __attribute__((aligned(16))) unsigned char lds[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & 3); // among the 4 waves that split the columns
    const int kgroup = KG == 2 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 8) : 0;
    const int g = lane >> 4, nl = lane & 15;
    int nb, m0;
    if (!take_block<ROWS, PACKED_K, DEVROWS>(p, nblocks_n, nblocks_m, lane, nb, m0)) return;
    if constexpr (KG == 2) {
        // (the launcher takes this form only for a K of a whole number of packed tiles per group)
        const int half_k = p.K / 2;
        p.packed += (size_t)kgroup * (half_k / PACKED_K) * 1024;
        p.A += (size_t)kgroup * half_k;
        p.K = half_k;
    }
    const int tile0 = __builtin_amdgcn_readfirstlane((nb * 4 + wave) * CT); // first 16-column tile of this wave

    // the tiles start at LDS offset 0 of the workgroup (the requests carry their LDS address in M0, all of it: the tiles of two K groups end at 128 KiB); behind them
    // the second group's row sums and NF4's table: byte -> {bf16 hi parts of (low, high) nibble, bf16 lo parts}
    uint2 *lut = (uint2 *)(lds + KG * NBUF * TILEB + (KG == 2 ? 2048 : 0));
    if constexpr (NF4) {
        if (threadIdx.x < 256) {
            const int i = threadIdx.x;
            const float c0 = c_nf4_big[i & 15], c1 = c_nf4_big[i >> 4];
            const uint32_t h0 = f32_to_bf16_ref(c0), h1 = f32_to_bf16_ref(c1);
            const uint32_t l0 = f32_to_bf16_ref(c0 - bf16_to_f32((uint16_t)h0));
            const uint32_t l1 = f32_to_bf16_ref(c1 - bf16_to_f32((uint16_t)h1));
            lut[i] = make_uint2(h0 | (h1 << 16), l0 | (l1 << 16));
        }
    }
    unsigned char *tiles = lds + kgroup * (NBUF * TILEB); // this group's

    f32x4 acc[CT][RT];
#pragma unroll
    for (int t = 0; t < CT; ++t)
#pragma unroll
        for (int m = 0; m < RT; ++m) acc[t][m] = f32x4 {0.f, 0.f, 0.f, 0.f};

    const int kt_n = __builtin_amdgcn_readfirstlane((p.K + KSTEP - 1) / KSTEP);
    // weights: the packed tile in scalar registers, a lane's chunk of it in one vector register; columns past the last tile read that one, unstored
    const XFT_GLOBAL uint8_t *wbase[CT];
#pragma unroll
    for (int t = 0; t < CT; ++t) {
        const int nt = tile0 + t < p.NTILES ? tile0 + t : p.NTILES - 1;
        wbase[t] = global_bytes((const uint8_t *)(uintptr_t)uniform_address(p.packed)) + (size_t)nt * __builtin_amdgcn_readfirstlane(p.KT) * 1024;
    }
    const uint32_t lane16 = lane * 16;
    u32x4 wreg[WSETS][WPARTS][CT];
    auto load_w = [&](int set, int kt_, int part, int t) {
        const int kt = kt_ < kt_n ? kt_ : kt_n - 1; // past the end: a valid tile, never used
        uint32_t at = lane16;
        asm volatile("" : "+v"(at)); // (or the compiler adds it to every tile's base ahead of the loop, a register pair each)
        wreg[set][part][t] = *(const XFT_GLOBAL u32x4 *)(wbase[t] + ((size_t)kt * (KSTEP / PACKED_K) + part) * 1024 + at);
    };

    // activations: request i of this wave fills LDS chunks 64 (ALOADS wave + i) ..+ 63 of a tile, a lane one of them, with the global chunk that belongs there
    uint32_t a_off[ALOADS]; // bytes
#pragma unroll
    for (int i = 0; i < ALOADS; ++i) {
        const int r = (64 / CPR) * (ALOADS * wave + i) + lane / CPR;
        int chunk = (lane % CPR) ^ direct_swizzle<KSTEP>(r);
        if (FOUR && p.K < KSTEP) chunk &= 7; // (64 k in all or in a part of K: both halves are those)
        int row = m0 + r;
        row = row < p.M ? row : p.M - 1;
        if constexpr (DEVROWS) row = p.a_rows ? p.a_rows[row] : row;
        a_off[i] = (uint32_t)row * (uint32_t)p.lda;
        asm volatile("" : "+v"(a_off[i])); // (or product and sum are one instruction with a register pair for its result, which the compiler then keeps)
        a_off[i] = (a_off[i] + chunk * 8) * 2;
    }
    // (Written as assembly: after the compiler's own builtin for this instruction it makes every later wait for a load or an LDS read a wait for all of them - an
    // instruction of the flat family that touches both memories.  Unaware of these requests, the compiler's counted waits for the weight loads come out a few
    // requests early, never late: the counter retires in order.  M0 carries the LDS address of the wave's first lane; one wait state between writing it and the
    // request.  The compiler holds nothing in M0 across statements.)
    const uint32_t lds_tiles = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)tiles + ALOADS * 1024 * wave;
    const uint16_t *a_uniform = (const uint16_t *)(uintptr_t)uniform_address(p.A);
    const int half_tail = FOUR ? __builtin_amdgcn_readfirstlane(p.K & 64) : 0; // 4-bit kinds: the last step has 64 k; requested with the 64 in front of them
    const int back = p.K < KSTEP ? 0 : half_tail;
    auto request_a = [&](int kt_, int i) {
        const int kt = kt_ < kt_n ? kt_ : kt_n - 1;
        const uint32_t dst = lds_tiles + (kt_ & (NBUF - 1)) * TILEB + i * 1024;
        const uint16_t *src = a_uniform + ((ptrdiff_t)kt * KSTEP - (kt == kt_n - 1 ? back : 0));
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(a_off[i]), "s"(src) : "memory");
    };

    // operands: lane (token nl, group g) reads one chunk of row nl of every row tile, 4 g + ms, 4 ms + g (BF16) or 2 g + ms (INT8)
    const int a_lane = nl * ROWB + (((FOUR ? 4 * g : BF16 ? g : 2 * g) ^ direct_swizzle<KSTEP>(nl)) << 4);
    auto a_at = [&](int ms) { return a_lane ^ ((BF16 ? 4 * ms : ms) << 4); };
    // NEED_SUM: wave w walks the row tiles in pairs, beginning with pair w, and sums the rows of its first two (RT = 6: the fourth wave those of the first) - no
    // branch on the wave number inside the k loop
    auto row_tile = [&](int m) { return NEED_SUM ? 2 * ((m / 2 + wave) % (RT / 2)) + (m & 1) : m; };
    MFrag afr[RT];
    auto read_a = [&](int buf, int ms, int m) { // buf: byte offset of the tile
        if constexpr (NEED_SUM)
            afr[m].q = *(const u32x4 *)(tiles + a_at(ms) + (buf + ((m / 2 + wave) % (RT / 2)) * (32 * ROWB)) + (m & 1) * (16 * ROWB));
        else
            afr[m].q = *(const u32x4 *)(tiles + a_at(ms) + buf + m * (16 * ROWB));
    };
    // UINT4: mask and exponent of a pair of codes in a scalar and a vector register of their own, so that they are one instruction (v_and_or_b32 takes no literal)
    uint32_t nib_mask = 0x000F000Fu, nib_bits = 0x43004300u;
    if constexpr (KIND == XFTHIP_W_UINT4) asm("" : "+s"(nib_mask), "+v"(nib_bits));
    auto widen = [&](int set, int ms, int t, MFrag &hi, MFrag &lo) {
        if constexpr (BF16) {
            hi.q = wreg[set][ms][t];
        } else if constexpr (KIND == XFTHIP_W_INT8) {
            const uint32_t x = wreg[set][0][t][2 * ms], y = wreg[set][0][t][2 * ms + 1];
            hi.u[0] = pack_hi16_m((float)(int)(int8_t)(x), (float)(int)(int8_t)(x >> 8));
            hi.u[1] = pack_hi16_m((float)(int)(int8_t)(x >> 16), (float)((int)x >> 24));
            hi.u[2] = pack_hi16_m((float)(int)(int8_t)(y), (float)(int)(int8_t)(y >> 8));
            hi.u[3] = pack_hi16_m((float)(int)(int8_t)(y >> 16), (float)((int)y >> 24));
        } else {
            const uint32_t x = wreg[set][0][t][ms];
            if constexpr (KIND == XFTHIP_W_UINT4) { // 0x4300 | u is the bf16 value 128 + u; the 128 is removed in the epilogue
                hi.u[0] = (x & nib_mask) | nib_bits;
                hi.u[1] = ((x >> 4) & nib_mask) | nib_bits;
                hi.u[2] = ((x >> 8) & nib_mask) | nib_bits;
                hi.u[3] = ((x >> 12) & nib_mask) | nib_bits;
            } else {
                const uint2 e0 = lut[x & 0xFF], e1 = lut[(x >> 8) & 0xFF], e2 = lut[(x >> 16) & 0xFF], e3 = lut[x >> 24];
                hi.u[0] = e0.x; hi.u[1] = e1.x; hi.u[2] = e2.x; hi.u[3] = e3.x;
                lo.u[0] = e0.y; lo.u[1] = e1.y; lo.u[2] = e2.y; lo.u[3] = e3.y;
            }
        }
    };
#define XFT_FENCE() __builtin_amdgcn_sched_barrier(0)
    // One step: the products of k tile kt, a group of RT MFMAs for each (32 k, column tile).  With them go the requests of activation tile kt + NBUF - 1, the loads of
    // weight tile kt + WD into the registers of the one that this step takes (4-bit: into the other set), the widening of the next group's weights and, behind the last
    // products that read it, the next activation operand.
    // The requests come in front of the loads: the compiler's wait for a tile's weights counts only the loads behind them, so that it is also one for as many of the
    // youngest requests.  With three tiles under way that leaves this step's out; in turn with them, and with two, each step waited for half of its own.  INT8, blocks alone
    // on their CUs, 500 x 4096 x 14336: 128 x 128 136 -> 106 us, with two K groups 91 -> 85, 128 x 256 156 -> 152; 600 x 4096 x 4096 33 -> 30.
    constexpr int WD = FOUR ? 1 : WSETS, AHEAD = NBUF - 1;
    constexpr int APG = FOUR ? 2 : (ALOADS + CT - 1) / CT; // requests a group that has some
    MFrag wcur_hi, wcur_lo;
    float rs[2] = {0.0f, 0.0f};
    constexpr int WREQS = CT * WPARTS; // weight loads a step, but for the steps behind the loop, whose loads nothing would take
    constexpr std::integral_constant<int, WREQS> loaded;
    constexpr std::integral_constant<int, 0> none;
    auto step = [&](int w_cur, int w_next, int w_load, int kt, auto loads) {
        const int buf = (kt & (NBUF - 1)) * TILEB, buf_next = ((kt + 1) & (NBUF - 1)) * TILEB;
#pragma unroll
        for (int ms = 0; ms < MICRO; ++ms) {
#pragma unroll
            for (int t = 0; t < CT; ++t) {
                const int q = ms * CT + t;
#pragma unroll
                for (int i = q * APG; i < (q + 1) * APG; ++i)
                    if (i < ALOADS) request_a(kt + AHEAD, i);
                if (FOUR && loads() && q >= ALOADS / 2 && q < ALOADS / 2 + CT) load_w(w_load, kt + WD, 0, q - ALOADS / 2);
                if (KIND == XFTHIP_W_INT8 && loads() && ms == 1) load_w(w_load, kt + WD, 0, t); // (its codes have been widened a group ago)
                MFrag nhi, nlo;
                if (t + 1 < CT) widen(w_cur, ms, t + 1, nhi, nlo);
                else if (ms + 1 < MICRO) widen(w_cur, ms + 1, 0, nhi, nlo);
                else widen(w_next, 0, 0, nhi, nlo);
                if constexpr (NEED_SUM) {
                    if (t == 0) {
                        typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
                        const bf16x2_t ones2 = __builtin_bit_cast(bf16x2_t, 0x3F803F80u);
#pragma unroll
                        for (int m = 0; m < 2; ++m)
#pragma unroll
                            for (int w = 0; w < 4; ++w) rs[m] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, afr[m].u[w]), ones2, rs[m], false);
                    }
                }
#pragma unroll
                for (int m = 0; m < RT; ++m) {
                    if constexpr (NF4) acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wcur_lo.v, afr[m].v, acc[t][m], 0, 0, 0);
                    acc[t][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wcur_hi.v, afr[m].v, acc[t][m], 0, 0, 0);
                    if (t == CT - 1 && (ms + 1 < MICRO || NBUF > 2)) {
                        if (ms + 1 < MICRO) read_a(buf, ms + 1, m);
                        else read_a(buf_next, 0, m);
                        __builtin_amdgcn_sched_barrier(0x6); // (each read behind the product that frees its registers; vector and scalar arithmetic may move)
                    }
                }
                wcur_hi = nhi;
                if constexpr (NF4) wcur_lo = nlo;
                XFT_FENCE();
                if (BF16 && loads()) load_w(w_load, kt + WD, ms, t);
            }
        }
    };
    int kt = 0;
    // prologue: the weight and activation tiles that the first step does not send
#pragma unroll
    for (int d = 0; d < WD; ++d) {
#pragma unroll
        for (int part = 0; part < WPARTS; ++part)
#pragma unroll
            for (int t = 0; t < CT; ++t) load_w(d, d, part, t);
#pragma unroll
        for (int i = 0; i < ALOADS; ++i)
            if (d < AHEAD) request_a(d, i);
    }
#pragma unroll
    for (int d = WD; d < AHEAD; ++d)
#pragma unroll
        for (int i = 0; i < ALOADS; ++i) request_a(d, i);
    XFT_FENCE();
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    widen(0, 0, 0, wcur_hi, wcur_lo);
    if constexpr (NBUF > 2) {
#pragma unroll
        for (int m = 0; m < RT; ++m) read_a(0, 0, m);
    }
    // Step k in weight set k % WSETS.  Four LDS tiles: the barrier that ends a step publishes the tile requested in the step before (everything but this step's own
    // requests and loads is in) and frees the one that this step read; the reads under way are of the next tile.  Two: it publishes the one requested in this step.
    // The counts are those of a step's own requests and loads, so that they hold only while the compiler leaves none of these loads out: behind the k loop the registers
    // that they fill are used once more, as far as it knows (kept).
    auto end_step = [&](auto loads) {
        XFT_FENCE();
        if constexpr (NBUF > 2) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(loads() + ALOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(loads()) : "memory");
        ++kt;
    };
    auto kept = [&](int sets) {
#pragma unroll
        for (int i = 0; i < sets; ++i)
#pragma unroll
            for (int part = 0; part < WPARTS; ++part)
#pragma unroll
                for (int t = 0; t < CT; ++t) asm volatile("" ::"v"(wreg[i][part][t]));
    };
#define XFT_STEP(s, loads)                                            \
    {                                                                 \
        step((s) % WSETS, ((s) + 1) % WSETS, (s) % WSETS, kt, loads); \
        end_step(loads);                                              \
    }
    if constexpr (FOUR) {
        auto one = [&](auto loads) { // (the next tile's registers are copied: 16 of them a step of 128 products)
#pragma unroll
            for (int m = 0; m < RT; ++m) read_a((kt & 1) * TILEB, 0, m);
            step(0, 1, 1, kt, loads);
            end_step(loads);
#pragma unroll
            for (int t = 0; t < CT && loads(); ++t) wreg[0][0][t] = wreg[1][0][t];
        };
        const int whole = kt_n - (half_tail ? 1 : 0);
        while (kt < whole) one(loaded);
        kept(1);
        if (half_tail) { // the last 64 k to their place, the k past the end count nothing
            for (int i = threadIdx.x & 255; i < ROWS * 8; i += 256) {
                const int r = i >> 3, c = i & 7;
                unsigned char *row = tiles + (kt & 1) * TILEB + r * ROWB;
                u32x4 *high = (u32x4 *)(row + (((8 + c) ^ direct_swizzle<KSTEP>(r)) << 4));
                *(u32x4 *)(row + ((c ^ direct_swizzle<KSTEP>(r)) << 4)) = *high;
                *high = u32x4 {0u, 0u, 0u, 0u};
            }
            __syncthreads();
            one(none);
        }
    } else {
        while (kt + WSETS <= kt_n) {
            XFT_STEP(0, loaded) XFT_STEP(1, loaded)
            if constexpr (WSETS > 2) XFT_STEP(2, loaded)
            if constexpr (WSETS > 3) XFT_STEP(3, loaded)
            if constexpr (WSETS > 4) XFT_STEP(4, loaded)
            if constexpr (WSETS > 5) XFT_STEP(5, loaded)
        }
        if (kt < kt_n) XFT_STEP(0, none)
        if (WSETS > 2 && kt < kt_n) XFT_STEP(1, none)
        if (WSETS > 3 && kt < kt_n) XFT_STEP(2, none)
        if (WSETS > 4 && kt < kt_n) XFT_STEP(3, none)
        if (WSETS > 5 && kt < kt_n) XFT_STEP(4, none)
    }
#undef XFT_STEP
#undef XFT_FENCE

    // ---- epilogue: lane holds columns 16 (tile0 + t) + 4 g .. + 3 of token m0 + 16 row_tile(m) + nl.  Each wave drops 32 rows of scaled results at a time, as fp32,
    // into an LDS patch of its own and walks it in 8-column chunks, consecutive lanes along a row (flush_rows)
    constexpr int OPITCH = 64 * CT + 16; // patch row pitch in bytes
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // the requests past the last tile have landed
    if constexpr (!FOUR) kept(WSETS);
    __syncthreads();                                 // every wave is past its last read of the activation tiles
    if constexpr (KG == 2) {
        // the second K group hands its accumulators over, 16 bytes a lane, from the start of LDS (at most the two groups' tiles), its row sums behind the tiles
        f32x4 *hand = (f32x4 *)lds + (size_t)wave * (CT * RT) * 64 + lane;
        float *hand_rs = (float *)(lds + KG * NBUF * TILEB) + wave * 128 + lane;
        if (kgroup == 1) {
#pragma unroll
            for (int t = 0; t < CT; ++t)
#pragma unroll
                for (int m = 0; m < RT; ++m) hand[(t * RT + m) * 64] = acc[t][m];
            if constexpr (NEED_SUM) hand_rs[0] = rs[0], hand_rs[64] = rs[1];
        }
        __syncthreads();
        if (kgroup == 0) {
#pragma unroll
            for (int t = 0; t < CT; ++t)
#pragma unroll
                for (int m = 0; m < RT; ++m) acc[t][m] += hand[(t * RT + m) * 64];
            if constexpr (NEED_SUM) rs[0] += hand_rs[0], rs[1] += hand_rs[64];
        }
        __syncthreads(); // (the result patches below overwrite what was handed over)
    }
    unsigned char *obuf = lds + wave * (32 * OPITCH);
    float sumA[RT];
    if constexpr (NEED_SUM) {
        // the lane groups hold quarters of a row's k range; every lane gets the sums of its tokens
        float *rowsum = (float *)(lds + 4 * 32 * OPITCH);
#pragma unroll
        for (int m = 0; m < 2; ++m) {
            float v = rs[m] + __shfl_xor(rs[m], 16, 64);
            v += __shfl_xor(v, 32, 64);
            if (g == 0 && kgroup == 0) rowsum[16 * row_tile(m) + nl] = v;
        }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < RT; ++m) sumA[m] = rowsum[16 * row_tile(m) + nl];
    }
    if (KG == 2 && kgroup == 1) return; // (no workgroup barrier from here on)
    const FlushRows to = flush_target(p, obuf, OPITCH, lane);
    f32x4 s[CT], z[CT];
#pragma unroll
    for (int t = 0; t < CT; ++t) {
        const int nt = tile0 + t < p.NTILES ? tile0 + t : p.NTILES - 1;
        s[t] = f32x4 {1.f, 1.f, 1.f, 1.f}, z[t] = f32x4 {0.f, 0.f, 0.f, 0.f};
        if constexpr (!BF16) s[t] = *(const f32x4 *)(p.scale + nt * 16 + 4 * g);
        if constexpr (KIND == XFTHIP_W_UINT4 || (KIND == XFTHIP_W_INT8 && NEED_SUM))
            if (p.zero) z[t] = *(const f32x4 *)(p.zero + nt * 16 + 4 * g);
    }
    auto value = [&](int t, int m, int e) {
        const float x = acc[t][m][e];
        if constexpr (KIND == XFTHIP_W_UINT4) return fmaf(s[t][e], x - 128.0f * sumA[m], z[t][e] * sumA[m]);
        else if constexpr (KIND == XFTHIP_W_INT8 && NEED_SUM) return fmaf(z[t][e], sumA[m], s[t][e] * x);
        else if constexpr (BF16) return x;
        else return s[t][e] * x;
    };
    float *put = (float *)(obuf + nl * OPITCH) + 4 * g;
    if (p.gateup) {
        // packed tiles alternate gate / up: a lane holds both of its output columns
        float bg[CT / 2][4], bu[CT / 2][4];
#pragma unroll
        for (int t = 0; t < CT; t += 2)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int col = (tile0 + t) * 8 + 4 * g + e;
                const bool there = p.bias && col < p.N / 2;
                bg[t / 2][e] = there ? p.bias[col] : 0.0f, bu[t / 2][e] = there ? p.bias[p.N / 2 + col] : 0.0f;
            }
#pragma unroll
        for (int m = 0; m < RT; ++m) {
#pragma unroll
            for (int t = 0; t < CT; t += 2) {
                f32x4 y;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float gate = value(t, m, e) + bg[t / 2][e], up = value(t + 1, m, e) + bu[t / 2][e];
                    y[e] = p.gateup == 2 ? clamped_glu(gate, up, p.glu_limit, p.glu_alpha) : up * silu_big(gate);
                }
                *(f32x4 *)(put + (m & 1) * (16 * OPITCH / 4) + 8 * t) = y;
            }
            if (m & 1) flush_rows<XFTHIP_EPI_NONE>(to, p, m0 + 16 * row_tile(m - 1), tile0 * 8, 8 * CT, p.N / 2);
        }
        return;
    }
    auto finish = [&](auto epi_tag) {
        constexpr int EPI = decltype(epi_tag)::value;
        float b[CT][4];
#pragma unroll
        for (int t = 0; t < CT; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int col = (tile0 + t) * 16 + 4 * g + e;
                b[t][e] = 0.0f;
                if constexpr (EPI == XFTHIP_EPI_BIAS || EPI == XFTHIP_EPI_RESIDENTIAL || EPI == XFTHIP_EPI_RESEXT) b[t][e] = p.bias && col < p.N ? p.bias[col] : 0.0f;
            }
#pragma unroll
        for (int m = 0; m < RT; ++m) {
#pragma unroll
            for (int t = 0; t < CT; ++t) {
                f32x4 y;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    float x = value(t, m, e);
                    if constexpr (EPI == XFTHIP_EPI_BIAS || EPI == XFTHIP_EPI_RESIDENTIAL || EPI == XFTHIP_EPI_RESEXT) x += b[t][e];
                    if constexpr (EPI == XFTHIP_EPI_SILU) x = silu_big(x);
                    if constexpr (EPI == XFTHIP_EPI_GELU) {
                        const float ex = fast_exp(1.702f * x);
                        x = ex / (ex + 1.0f) * x;
                    }
                    y[e] = x; // the residual operand joins in flush_rows
                }
                *(f32x4 *)(put + (m & 1) * (16 * OPITCH / 4) + 16 * t) = y;
            }
            if (m & 1) flush_rows<EPI>(to, p, m0 + 16 * row_tile(m - 1), tile0 * 16, 16 * CT, p.N);
        }
    };
    switch (p.epi) {
        case XFTHIP_EPI_BIAS: finish(std::integral_constant<int, XFTHIP_EPI_BIAS> {}); break;
        case XFTHIP_EPI_SILU: finish(std::integral_constant<int, XFTHIP_EPI_SILU> {}); break;
        case XFTHIP_EPI_GELU: finish(std::integral_constant<int, XFTHIP_EPI_GELU> {}); break;
        case XFTHIP_EPI_RESMUL: finish(std::integral_constant<int, XFTHIP_EPI_RESMUL> {}); break;
        case XFTHIP_EPI_RESIDENTIAL: finish(std::integral_constant<int, XFTHIP_EPI_RESIDENTIAL> {}); break;
        case XFTHIP_EPI_RESEXT: finish(std::integral_constant<int, XFTHIP_EPI_RESEXT> {}); break;
        default: finish(std::integral_constant<int, XFTHIP_EPI_NONE> {}); break;
    }
}

template <int KIND, int CT, int RT, bool NEED_SUM, bool DEVROWS, int KG>
static int launch_direct(const SkinnyParams &p, hipStream_t stream) {
    using T = DirectTraits<KIND, CT, KG>;
    BlockGrid g;
    if (int rc = block_grid<DEVROWS>(p, 16 * RT, 4 * CT, g)) return rc;
    // the activation tiles, the second K group's row sums and NF4's table; reused after the k loop by the four waves' output patches and the row sums
    const size_t pipe = (size_t)KG * T::NBUF * 16 * RT * T::KSTEP * 2 + (KG == 2 ? 2048 : 0) + (KIND == XFTHIP_W_NF4 ? 2048 : 0);
    const size_t patches = 4 * 32 * (64 * CT + 16) + 16 * RT * sizeof(float), smem = pipe > patches ? pipe : patches;
    if (smem > 64 * 1024) { // more dynamic LDS than the default limit: raise it once per instantiation
        static const hipError_t attr = hipFuncSetAttribute((const void *)qgemm_direct_kernel<KIND, CT, RT, NEED_SUM, DEVROWS, KG>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        XFT_CHECK_HIP(attr);
    }
    SkinnyParams q = p;
    q.band = g.band;
    hipLaunchKernelGGL((qgemm_direct_kernel<KIND, CT, RT, NEED_SUM, DEVROWS, KG>), dim3(g.blocks), dim3(256 * KG), smem, stream, q, g.nblocks_n, g.nblocks_m);
    XFT_CHECK_HIP(hipGetLastError());
    return 0;
}

} // namespace
} // namespace xfthip
