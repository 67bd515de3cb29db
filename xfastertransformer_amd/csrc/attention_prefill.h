// Prefill attention: many (query token, query head) columns per (sequence, KV head).
//
// Replaces the reference's flash-style prefill (xft::selfScaledDpAttention, src/kernels/attention_kernels.h:1283-1408;
// DecoderUtil::incrementalTileAttention / softmaxTile / updateOutTile, src/utils/decoder_util.h:606-889) and its
// chunked prefill over a cache (xft::crossAttnByHead, attention_kernels.h:988-1123) when a launch has enough
// columns to fill the device.
//
// A workgroup shares each 32-token block of keys and values through LDS; a wave owns 32 columns.
//
//   S^T = K . Q^T   32 tokens (rows) x 32 columns; A = keys from LDS, B = the wave's queries, held in registers for the whole walk
//   O^T += V^T . P^T  128 dims x 32 columns; A = values from LDS (token index innermost, as the cache
//                   stores them), B = probabilities straight from the score registers
//
// Two forms.  In 32 x 32 x 16 MFMAs one operand read from LDS is one MFMA; a lane owns one column and 16 of a block's tokens (8 q + 4 h + s; h = lane / 32, q = 0..3,
// s = 0..3).  FINE, in 16 x 16 x 32 ones: two column tiles, an operand read is two MFMAs; a lane owns two columns and 8 tokens (16 tt + 4 g + r; g = lane / 16).
// The same products take less of the card's power as 16 x 16 x 32, and more instructions.
// The cache stores a value block with its tokens permuted (kvcache.h: 16-byte chunk c of a dim row = tokens 4 c .. 4 c + 3 and 16 + 4 c .. 16 + 4 c + 3): chunk
// c = 2 t + h is what lane half h holds in registers q = t and q = t + 2, chunk g what lane group g holds of its two score tiles, so that the probabilities are the B
// operand of the values without an exchange between lanes.
//
// Online softmax per column in the log2 domain, fp32; the reference point moves only when a block's maximum
// exceeds it by more than 2^8 (probabilities up to 256 are exact enough in fp16 and in the fp32 sums), so the
// 64 accumulator registers of a lane are rescaled in few blocks only.
//
// Four waves a workgroup, two workgroups a CU.  INT8 cache: codes are widened to fp16 (exact) on their way into LDS, the key scale multiplies
// the score row, the value scale the probability; the value scales are taken relative to a running reference that moves lazily, too (when a
// block's largest scale leaves [ref / 1024, 4 ref]), so fp16 probabilities stay in range whatever the scales.
#pragma once
#include <type_traits>

#include "attention_dev.h"

namespace xfthip {

union HFrag32 {
    f16x8 v;
    uint32_t u[4];
    u32x4 q;
};

__device__ inline f32x16 prefill_mfma(const f16x8 a, const f16x8 b, const f32x16 c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
__device__ inline f32x4 prefill_mfma(const f16x8 a, const f16x8 b, const f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }

// a lane's column: dims 32 dt + 8 q + 4 h .. (FINE: 16 dt + 4 g ..)
template <typename Acc, int DT>
__device__ inline void store_direct(const AttnParams &p, const size_t base, const int part, const Acc (&o)[DT], const float inv) {
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int q = 0; q < (DT == 8 ? 1 : 4); ++q) {
            const size_t idx = base + 128 / DT * dt + 8 * q + 4 * part;
            const float v0 = o[dt][4 * q] * inv, v1 = o[dt][4 * q + 1] * inv, v2 = o[dt][4 * q + 2] * inv, v3 = o[dt][4 * q + 3] * inv;
            if (p.out_dtype == XFTHIP_BF16) {
                const uint32_t lo = f32x2_to_bf16(v0, v1), hi = f32x2_to_bf16(v2, v3);
                uint16_t *dst = (uint16_t *)p.out + idx;
                if ((((uintptr_t)dst) & 7) == 0) {
                    *(uint2 *)dst = make_uint2(lo, hi);
                } else {
                    dst[0] = (uint16_t)lo, dst[1] = (uint16_t)(lo >> 16), dst[2] = (uint16_t)hi, dst[3] = (uint16_t)(hi >> 16);
                }
            } else {
                float *dst = (float *)p.out + idx;
                dst[0] = v0, dst[1] = v1, dst[2] = v2, dst[3] = v3;
            }
        }
}

// LDS rows are 64 bytes; the 16-byte chunk c of row r lies in slot c ^ row_turn(r).  A FINE operand read is rows 0 .. 15, chunk g of lane group g; its lanes are served 16 at a
// time, not always neighbours: 0 .. 3 and 12 .. 15 of one group go with 4 .. 11 of the next, whose chunk differs in bit 0.  So rows of the two kinds differ in bit 1.
template <bool FINE>
__device__ inline int row_turn(int r) {
    if constexpr (!FINE) return (r >> 2) & 3;
    return (((r >> 2) ^ (r >> 3)) & 1) << 1 | ((r >> 3) & 1);
}

// Workgroups are handed to the 8 XCDs in turn by their linear index, and each XCD has an L2 of its own: the (sequence, KV head) pairs are dealt to the
// XCDs (pair = 8 group + XCD).  An XCD takes its groups in bands of five, and the column groups of a band's pairs in turn, longest history first: what
// runs at the end is short then.  Pair after pair instead, an XCD ended on the long walks of its last pair wherever its 64 workgroups at a time were
// no multiple of the pairs' own: 5 x 700 tokens, 32 query / 8 KV heads 47 -> 41 us, 2 x 2000, 32 / 32 heads 123 -> 102, 5 x 1500 INT8 236 -> 197, 4 x 2000, 32 / 8
// heads INT8 213 -> 206, FP16 153 in either order (63 column groups fill the 64 places).  96 FP16 shapes of 1 to 12 sequences, 16 .. 64 / 4 .. 32 heads: 0.97 of the time in the geometric
// mean, with one query head a KV head 0.90, four 0.94, six 0.99, eight and sixteen, whose pairs have many column groups, the same (0.95 .. 1.055, as the runs differ); 70 INT8 0.93, 36
// paged 0.98.  Bands of 4 and 6: within 0.1 % of that in 31 shapes; of 3 or of 16 1 to 2 % slower (8 x 800 tokens 57.5 -> 60.0, 8 x 3900, 32 / 32 heads, in one 1161 -> 1353: an L2 does not hold that many pairs' keys and values).
constexpr int kBand = 5;
struct PrefillBands { // what is left of whole bands comes first, `rest` groups; then bands of `width`
    int rest, width;
};
inline PrefillBands prefill_bands(const int groups) { return {groups % kBand, kBand}; }
// the band of a group
__host__ __device__ inline void prefill_band(const PrefillBands b, const int group, int &first, int &width) {
    const bool whole = group >= b.rest;
    width = whole ? b.width : b.rest, first = whole ? b.rest + (group - b.rest) / b.width * b.width : 0;
}

// 128 columns a workgroup.  Figures are those of the FP16 cache where nothing else is said.
//
// A wave's time on a block of 32 tokens is the product phase - scores of block b + 1 and values of block b, 16 MFMAs of 32 x 32 (512 clocks; FINE 32 of 16 x 16), and behind each the
// read of the operand that takes its place: keys of block b + 2, values of block b + 1 - and the softmax phase, the probabilities of the block's scores, about 90
// vector instructions, 16 of them exponentials, and the request of block b + kLook.  The two waves of a SIMD, of two workgroups, share its matrix unit
// and vector ALU; products go first (s_setprio: 5 % slower without).  Reading all operands of a block in front of its products kept the wave from issuing
// them, and every vector instruction of one wave - a sum of probabilities, an address, a result's narrowing - is time the other does not get:
// against that form 4 x 2000 tokens, 32 query / 8 KV heads, 179 -> 152 us (145 back to back, 905 TFLOP/s), 12 x 200 tokens 27 -> 22.  Matrix unit and
// vector ALU are busy 45 and 43 % of the clocks (INT8 27 and 60), the issue of MFMAs counted with the latter.  Tried and not kept:
// half of the exponentials between the MFMAs (an exponential holds up the other wave's MFMAs: 8 % slower), operands read in the softmax phase (6 %), scores and values
// in turn (the same), the scale in the queries and the reference point as the score's initial value (the same, and the queries lose bits).
// Eight waves a workgroup that share a block and take turns at the matrix unit behind barriers: 1450 clocks a block instead of
// about 2300 a pair of waves, but 3 us in front of the walk, 2.6 behind it and as much until the next workgroup began, in which the CU does nothing
// else: 150 - 170 us for the first, 23 for the second of the calls above; with workgroups that stay, the next columns' blocks and queries on their way while these
// are walked, 146 and 34, the change from one to the next being worth four blocks.
//
// LDS: a ring of four 32-token blocks, 8 KB of keys and 8 KB of values each, which go global -> LDS without a stop in registers
// (global_load_lds_dwordx4: a wave instruction fills 1 KiB of consecutive LDS, lane after lane, from 64 addresses of its
// choice; wave w requests the w-th 2 KiB of both).  Keys lie as four segments of 32 dims, values as they lie in the cache: rows of 64
// bytes, the 16-byte chunk c of row r in slot c ^ ((r >> 2) & 3), which keeps the operand reads (32 rows, one chunk index) free of
// bank conflicts and leaves each of them one of two addresses and a constant.  In front of the walk the ring's upper half holds the queries, behind it
// the ring the results, so that both travel as whole rows.
// (The requests as assembly: after the compiler's builtin for this instruction every later counted wait becomes a wait for
// everything.  M0 carries the LDS address of the wave's first lane; one wait state between writing it and the request.)
//
// INT8: the blocks go through registers, a block ahead, where they are widened: 40 vector instructions more a block and wave, and 50 for the scales and
// the sums of probabilities that are other numbers than those multiplied.  That wants no request in flight, so three blocks of ring are enough, and
// the queries are read straight into registers, unscaled (the key scales are in fp32 anyway).  Call with the append, 32 query / 8 KV heads, against two
// buffers whose operands were all read in front of the products: 4 x 2000 tokens 264 -> 218 us, 12 x 200 41 -> 30, 2 x 700 behind 1900 134 -> 110; with 32
// KV heads 360 -> 300, 57 -> 46, 148 -> 130.  Measured and not kept: the block in LDS as codes, widened by every wave (354 us for 4 x 2048).
//
// FP16: the queries carry the power of two in the softmax scale, the rest of it multiplies the scores in fp32: a bf16 value is exact in fp16 from 2^-17 / that
// power up to 65504 / it.  Of a scale below 2^-4 / log2 e they carry a power of two of their own.  Where `plain` is set, they carry nothing, as in the form for few columns.  The row sums are those of the rounded probabilities.
//
// Which form.  FINE where the launch runs for so long that the card's power bounds it (4 x 2000 tokens: 168 us in 32 x 32 MFMAs, 125 where all operands are zeros); else its instructions, twice as many MFMAs and exchanges, cost more than its power saves.
// FP16, mean workgroups x blocks of 32 tokens a CU in brackets, us of the call: 4 x 2000 tokens, 32 / 8 heads (250) 168 -> 160, 1 x 4000 (240) 136 -> 127, 2 x 2000, 32 / 32
// (125) 104 -> 99, 8 x 1000 (125) 97 -> 94, paged 6 x 1500 (120) 112 -> 111, 2 x 2800, 32 / 32 (190) 165 -> 158; but 3 x 1200, 32 / 32 (70) 73 -> 72, 2 x 700 behind 1900
// (97, 1.4 workgroups a CU) 73 -> 73, 4 x 800 (40) 40 -> 42, 8 x 500 (30) 37 -> 40, 512 behind 8000, half a workgroup a CU, 153 -> 154.
// INT8, mean tokens walked in brackets: 4 x 2000 (1000) 226 -> 217, 5 x 1500 (750) 157 -> 148, 2 x 3500, 32 / 32 (1750) 344 -> 322, 512 behind 8000 (8250) 295 -> 282,
// 900 (450) 40.2 -> 39.4; but 8 x 400 (200) 37.0 -> 37.7, 12 x 200 (100) 28.7 -> 28.8.
// walk: the tokens that a column sees on average; least: blocks a CU from which on FP16 takes it
inline bool prefill_fine(bool int8, long workgroups, long walk, long least = 80) {
    const long cus = device_cu_count();
    return int8 ? walk >= 256 : workgroups >= 2 * cus && workgroups * (walk / 32) >= least * cus;
}
// S new tokens behind `past` for each of `pairs` (sequence, KV head) pairs, G query heads a KV head: 0 the form for few columns, 1 this one, 2 this one, FINE.  This one (a wave walks the
// whole visible sequence for its 32 columns) is taken once waves of 16 columns would fill the device.
inline int attention_prefill_form(bool int8, int G, long pairs, int S, int past) {
    if (S <= 1 || pairs * ((S * G + 15) / 16) < 4L * device_cu_count()) return 0;
    return prefill_fine(int8, pairs * ((S * G + 127) / 128), past + S / 2) ? 2 : 1;
}

constexpr int kRing = 4, kLook = kRing - 1, kRingBlock = 16384, kRingLds = kRing * kRingBlock;
constexpr int kScaleBytes = 256; // 32 key scales and 32 value scales of a block
constexpr int kRingLdsInt8 = 3 * (kRingBlock + kScaleBytes);

// lds: kRingLds or kRingLdsInt8 bytes; every thread of 256 calls it.  plain (FP16): the queries as they are
template <bool INT8, bool FINE>
__device__ inline void attn_prefill_ring_unit(const AttnParams &p, const int kvh, const int cgroup, const int b, unsigned char *lds, const bool plain = false) {
    constexpr int D = 128, NW = 4, WC = 32;
    // column tiles a wave, their columns, score and value accumulators a column tile, k-steps of the scores; a lane's scores of a column and accumulators' registers
    constexpr int CT = FINE ? 2 : 1, TW = 32 / CT, XT = FINE ? 2 : 1, DT = FINE ? 8 : 4, QS = FINE ? 4 : 8, V = 16 / CT, AL = V / XT;
    using Acc = std::conditional_t<FINE, f32x4, f32x16>;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int h = lane >> 5, cl = lane & 31, part = lane / TW, tl = lane % TW;
    int past = p.past;
    if (p.past_dev) {
        past = p.past_dev[b];
        past = past < 0 ? 0 : (past > p.kv.S - p.S ? p.kv.S - p.S : past);
    }
    past = __builtin_amdgcn_readfirstlane(past);
    const int ncols = p.S * p.G;
    const int c0 = (cgroup * NW + wave) * WC; // first column of this wave
    const int c = c0 + cl;
    const bool cvalid = c < ncols;
    const int cs = cvalid ? c / p.G : 0, cj = cvalid ? c % p.G : 0;
    // (c: the column whose rows of queries and results this lane finds; its products are of columns c0 + TW ct + tl)
    int limit[CT]; // tokens [0, limit) are visible to that column, if there is one
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) limit[ct] = FINE ? __shfl(cvalid ? past + cs + 1 : 0, TW * ct + tl, 64) : cvalid ? past + cs + 1 : 0;
    auto token = [&](int r) { return (FINE ? 16 : 8) * (r >> 2) + 4 * part + (r & 3); }; // of score r of a column, in its block
    const int lim_min = c0 + WC - 1 < ncols ? past + c0 / p.G + 1 : 0; // every column of the wave sees at least this many
    const int wave_last = c0 + WC - 1 < ncols ? c0 + WC - 1 : ncols - 1;
    const int wave_lim = c0 < ncols ? past + wave_last / p.G + 1 : 0, wave_nblk = (wave_lim + 31) >> 5; // no column of the wave sees a token from here on
    const int wg_last = (cgroup + 1) * NW * WC - 1 < ncols ? (cgroup + 1) * NW * WC - 1 : ncols - 1;
    const int nblk = (past + wg_last / p.G + 1 + 31) >> 5;
    const size_t bh = (size_t)b * p.kv.H + kvh;
    auto slot = [](const int blk) { return INT8 ? blk % 3 : blk & (kRing - 1); };
    auto sgpr_ptr = [](const void *ptr) { // the same in every lane; said so, for a scalar register pair
        const uint64_t bits = (uint64_t)(uintptr_t)ptr;
        return (const char *)(uintptr_t)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(bits >> 32)) << 32) |
                (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)bits));
    };
    constexpr int ESZ = INT8 ? 1 : 2, BLOCK = 32 * D * ESZ; // bytes of a cached value, of a block's keys
    const char *k_uniform = sgpr_ptr((const char *)p.kv.k + bh * p.kv.S * D * ESZ), *v_uniform = sgpr_ptr((const char *)p.kv.v + bh * p.kv.S * D * ESZ);

    // ---- requests: this wave's share of a block is key segment w and dims 32 w .. of the values ----
    uint32_t rq_koff[2], rq_voff[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const int kr = 16 * i + (lane >> 2), vr = 32 * wave + 16 * i + (lane >> 2);
        rq_koff[i] = kr * 256 + wave * 64 + (((lane & 3) ^ row_turn<FINE>(kr)) << 4);
        rq_voff[i] = vr * 64 + (((lane & 3) ^ row_turn<FINE>(vr)) << 4);
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds;
    auto request = [&](const int blk_raw) {
        const int blk = __builtin_amdgcn_readfirstlane(blk_raw < nblk ? blk_raw : nblk - 1); // (past the end: the last block again, never read as itself)
        const char *ks = k_uniform + (size_t)blk * BLOCK, *vs = v_uniform + (size_t)blk * BLOCK;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t kd = lds0 + 2048 * (uint32_t)wave + 1024 * i + (blk_raw & (kRing - 1)) * kRingBlock, vd = kd + 8192;
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(kd), "v"(rq_koff[i]), "s"(ks) : "memory");
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(vd), "v"(rq_voff[i]), "s"(vs) : "memory");
        }
    };
    // ---- INT8: a thread's 16 codes of a block's keys and of its values, by way of registers, where they are widened (exact) ----
    // (eight lanes write eight rows of a segment, which fall on different banks)
    const ATTN_GLOBAL float *scales = (const ATTN_GLOBAL float *)(h ? p.kv.vscale : p.kv.kscale) + bh * p.kv.S + cl;
    const int ck = lane >> 3, tk = 8 * wave + (lane & 7), vd = 32 * wave + cl; // 16 dims 16 ck .. of token tk; token slots 16 h .. of dim vd
    u32x4 kstage, vstage;
    float sstage; // wave 0: a key or value scale a lane
    auto fetch = [&](const int blk) {
        kstage = *(const ATTN_GLOBAL u32x4 *)(const ATTN_GLOBAL char *)(k_uniform + (size_t)blk * BLOCK + tk * D + 16 * ck);
        vstage = *(const ATTN_GLOBAL u32x4 *)(const ATTN_GLOBAL char *)(v_uniform + (size_t)blk * BLOCK + vd * 32 + 16 * h);
        if (wave == 0) sstage = scales[blk << 5];
    };
    auto stash = [&](const int blk) {
        unsigned char *block = lds + slot(blk) * kRingBlock;
        auto put = [](unsigned char *row, const int c, const int turn, const u32x4 raw) { // chunks c and c + 1 of a row
            HFrag32 lo, hi;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                h2 a, b;
                widen_i8x4(raw[i], a, b);
                lo.u[2 * i] = __builtin_bit_cast(uint32_t, a), lo.u[2 * i + 1] = __builtin_bit_cast(uint32_t, b);
                widen_i8x4(raw[2 + i], a, b);
                hi.u[2 * i] = __builtin_bit_cast(uint32_t, a), hi.u[2 * i + 1] = __builtin_bit_cast(uint32_t, b);
            }
            *(u32x4 *)(row + ((c ^ turn) << 4)) = lo.q;
            *(u32x4 *)(row + (((c + 1) ^ turn) << 4)) = hi.q;
        };
        put(block + (ck >> 1) * 2048 + tk * 64, 2 * (ck & 1), row_turn<FINE>(tk), kstage);
        put(block + 8192 + vd * 64, 2 * h, row_turn<FINE>(vd), vstage);
        if (wave == 0) *(float *)(lds + 3 * kRingBlock + slot(blk) * kScaleBytes + 4 * lane) = sstage;
    };
    if constexpr (INT8) {
        fetch(0);
    } else {
        request(0);
        request(1);
    }

    // ---- this wave's queries: B operand of the score MFMA, k-step s covers dims 128 / QS s + 8 part .. + 8 of column TW ct + tl ----
    float c1[CT], qmul[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) c1[ct] = p.scale * 1.4426950408889634f, qmul[ct] = 1.0f;
    HFrag32 qf[CT][QS];
    auto take_query = [&](const int ct, const int s, const u32x4 raw) {
#pragma unroll
        for (int i = 0; i < 4; ++i) qf[ct][s].u[i] = pack_f16(u2f(raw[i] << 16) * qmul[ct], u2f(raw[i] & 0xFFFF0000u) * qmul[ct]);
    };
    // FP16: through the ring's upper half
    unsigned char *qbuf = lds + (kRing / 2) * kRingBlock + wave * 8192;
    const uint64_t qrow = (uint64_t)(uintptr_t)(p.q + ((size_t)b * p.S + cs) * p.qStride + (size_t)(kvh * p.G + cj) * D);
    auto of_column = [&](uint64_t mine, int r) { // the 64 bits that column r of the wave holds
        return (uint64_t)(uint32_t)__shfl((int)(uint32_t)mine, r, 64) | ((uint64_t)(uint32_t)__shfl((int)(mine >> 32), r, 64) << 32);
    };
    if constexpr (!INT8) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int r = 4 * i + (lane >> 4); // the 16-byte chunk c of a row sits in slot c ^ (row & 15)
            const uint64_t src = of_column(qrow, r) + (((lane & 15) ^ (r & 15)) << 4);
            const uint32_t dst = lds0 + (kRing / 2) * kRingBlock + 8192 * (uint32_t)wave + i * 1024;
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(dst), "v"(src) : "memory");
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        auto query = [&](const int ct, const int s) { return *(const u32x4 *)(qbuf + (TW * ct + tl) * 256 + (((16 / QS * s + part) ^ (tl & 15)) << 4)); };
        const float two = u2f(f2u(c1[0]) & 0x7F800000u);
        if (!plain && two <= 1.0f) {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) qmul[ct] = two;
            if (two < 0.0625f) {
                // A scale that small would push ordinary queries among fp16's subnormal values: the power of two that takes the column's own largest value to 2^13 or more
                // instead (a real branch)
                asm volatile("" ::: "memory");
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) {
                    uint32_t top = 0; // its exponent
#pragma unroll
                    for (int s = 0; s < QS; ++s) {
                        const u32x4 raw = query(ct, s);
#pragma unroll
                        for (int i = 0; i < 4; ++i) top = max(top, max(raw[i] << 1 >> 24, raw[i] << 17 >> 24));
                    }
                    if constexpr (FINE) top = max(top, (uint32_t)__shfl_xor((int)top, 16, 64));
                    top = max(top, (uint32_t)__shfl_xor((int)top, 32, 64));
                    qmul[ct] = u2f((267u - min(max(top, 14u), 254u)) << 23);
                }
            }
        }
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            c1[ct] /= qmul[ct];
#pragma unroll
            for (int s = 0; s < QS; ++s) take_query(ct, s, query(ct, s));
        }
    } else {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            const uint64_t row = FINE ? of_column(qrow, TW * ct + tl) : qrow; // (past the last column: the first one's)
#pragma unroll
            for (int s = 0; s < QS; ++s) take_query(ct, s, *(const u32x4 *)((const uint16_t *)(uintptr_t)row + 128 / QS * s + 8 * part));
        }
    }

    const h2 ones2 = {(_Float16)1.0f, (_Float16)1.0f};
    float m_run[CT], l_run[2] = {0.0f, 0.0f}; // a column's reference point; sums of this lane's rows, of the two columns or, in turn, of the one
    float vref = 0.0f; // INT8: the value scales are taken relative to this (0 = not set yet)
    unsigned long long unset[CT]; // lanes whose column has seen nothing above minus infinity yet
    Acc o[CT][DT], x[CT][XT]; // x: the scores
    HFrag32 kf[8], vf[8], pf[2];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        m_run[ct] = 0.0f, unset[ct] = ~0ull;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int r = 0; r < AL; ++r) o[ct][dt][r] = 0.0f;
    }
    // operand addresses: one of two (which half of a 64-byte row; FINE: the same), the rest constants
    const uint32_t at0 = tl * 64 + ((part ^ row_turn<FINE>(tl)) << 4), at1 = FINE ? at0 : tl * 64 + (((2 + part) ^ row_turn<FINE>(tl)) << 4);
    // operand i of a block's keys (k-step i; FINE: k-step i / 2, token tile i % 2), of its values (k-step i / 4, dim tile i % 4; FINE: dim tile i)
    auto key_at = [&](const int i) { return FINE ? at0 + (i >> 1) * 2048 + (i & 1) * 1024 : (i & 1 ? at1 : at0) + (i >> 1) * 2048; };
    auto value_at = [&](const int i) { return FINE ? at0 + i * 1024 : (i >> 2 ? at1 : at0) + (i & 3) * 2048; };
    auto across = [](float v) { // the largest of the lanes that share a column
        if constexpr (FINE) v = fmaxf(v, swap16(v));
        return fmaxf(v, swap32(v));
    };
    auto scale_all = [&](const int ct, const float by) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int r = 0; r < AL; ++r) o[ct][dt][r] *= by;
    };

    auto softmax = [&](const int blk) {
        const int t0 = blk << 5;
        const float *sl = (const float *)(lds + 3 * kRingBlock + slot(blk) * kScaleBytes); // INT8: key scales, value scales
        auto score = [&](const int ct, const int r) -> float { return x[ct][r / AL][r % AL]; };
        auto set_score = [&](const int ct, const int r, const float v) { x[ct][r / AL][r % AL] = v; };
        if constexpr (INT8) {
#pragma unroll
            for (int q = 0; q < V / 4; ++q) {
                const f32x4 ks = *(const f32x4 *)(sl + token(4 * q)) * c1[0]; // key scale and softmax scale in one factor (of every column)
#pragma unroll
                for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                    for (int r = 0; r < 4; ++r) set_score(ct, 4 * q + r, fmaf(score(ct, 4 * q + r), ks[r], -m_run[ct]));
            }
        } else {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int r = 0; r < V; ++r) set_score(ct, r, fmaf(score(ct, r), c1[ct], -m_run[ct]));
        }
        if (t0 + 32 > lim_min) {
            // only the blocks on the causal diagonal pay for the mask (a real branch)
            asm volatile("" ::: "memory");
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int r = 0; r < V; ++r) set_score(ct, r, t0 + token(r) < limit[ct] ? score(ct, r) : kNegBig);
        }
        // x = log2-domain score minus the column's reference point (0 while the column has seen nothing)
        float bmax[CT];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
            bmax[ct] = fmaxf(fmaxf(score(ct, 0), score(ct, 1)), score(ct, 2));
#pragma unroll
            for (int r = 3; r < V - 1; r += 2) bmax[ct] = fmaxf(fmaxf(bmax[ct], score(ct, r)), score(ct, r + 1));
            bmax[ct] = fmaxf(bmax[ct], score(ct, V - 1));
        }
        // the reference point moves when the block's maximum exceeds it by more than 2^8, and is set by the
        // first block a column sees anything of
        if ((__builtin_amdgcn_ballot_w64(fmaxf(bmax[0], bmax[CT - 1]) > 8.0f) | unset[0] | unset[CT - 1]) != 0) {
            // a real branch: in most blocks no column of the wave moves
            asm volatile("" ::: "memory");
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) {
                const float top = across(bmax[ct]);
                const bool fresh = (unset[ct] >> lane) & 1, set = fresh && top > 0.5f * kNegBig, move = set || top > 8.0f;
                const float delta = move ? top : 0.0f, alpha = set ? 1.0f : __builtin_amdgcn_exp2f(-delta); // (a column that sees its first tokens holds zeros)
                unset[ct] = __builtin_amdgcn_ballot_w64(fresh && !set && limit[ct] > 0);
                m_run[ct] += delta;
                l_run[ct] *= alpha;
                if constexpr (!FINE) l_run[1] *= alpha;
#pragma unroll
                for (int r = 0; r < V; ++r) set_score(ct, r, score(ct, r) - delta);
                scale_all(ct, alpha);
            }
        }
        float pr[CT][V];
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int r = 0; r < V; ++r) pr[ct][r] = __builtin_amdgcn_exp2f(score(ct, r)); // (a masked score is kNegBig: 0)
        if constexpr (INT8) {
            // (the sums are those of the probabilities as they are: with the scales and rounded, they are other numbers)
#pragma unroll
            for (int ct = 0; ct < CT; ++ct)
#pragma unroll
                for (int r = 0; r < V; r += 4) l_run[FINE ? ct : r >> 2 & 1] += (pr[ct][r] + pr[ct][r + 1]) + (pr[ct][r + 2] + pr[ct][r + 3]);
            __builtin_amdgcn_sched_barrier(0); // (the scales' registers only now)
            f32x4 vs[V / 4];
            float vmax = 0.0f;
#pragma unroll
            for (int q = 0; q < V / 4; ++q) vs[q] = *(const f32x4 *)(sl + 32 + token(4 * q));
            if (t0 + 32 > wave_lim) {
                // tokens no column of the wave sees stay out: behind the sequence's end the cache may hold anything (a real branch)
                asm volatile("" ::: "memory");
#pragma unroll
                for (int r = 0; r < V; ++r) vs[r >> 2][r & 3] = t0 + token(r) < wave_lim ? vs[r >> 2][r & 3] : 0.0f;
            }
#pragma unroll
            for (int r = 0; r < V; r += 2) vmax = fmaxf(fmaxf(vmax, vs[r >> 2][r & 3]), vs[r >> 2][(r & 3) + 1]);
            vmax = across(vmax); // the block's largest value scale, the same in every lane
            // value scales relative to vref; vref follows the blocks' largest scale lazily, like the maximum
            if (vmax > 4.0f * vref || (vmax > 0.0f && vmax * 1024.0f < vref)) { // wave-uniform
                asm volatile("" ::: "memory");
                const float vmove = vref > 0.0f ? vref / vmax : 1.0f;
                vref = vmax;
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) scale_all(ct, vmove);
            }
            const float vinv = vref > 0.0f ? 1.0f / vref : 0.0f;
#pragma unroll
            for (int r = 0; r < V; ++r) {
                const float by = vs[r >> 2][r & 3] * vinv;
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) pr[ct][r] *= by;
            }
        }
#pragma unroll
        for (int t = 0; t < 2; ++t) // k-step or column t of the values' products
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int ct = FINE ? t : 0, r = FINE ? 2 * i : 4 * t + 2 * (i & 1) + 8 * (i >> 1);
                pf[t].u[i] = pack_f16(pr[ct][r], pr[ct][r + 1]);
            }
        if constexpr (!INT8) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int i = 0; i < 4; ++i) l_run[FINE ? t : i & 1] = __builtin_amdgcn_fdot2(__builtin_bit_cast(h2, pf[t].u[i]), ones2, l_run[FINE ? t : i & 1], false);
        }
    };
    // scores of block `next` (keys already read), values of the block in front of it; reads the keys of block next + 1, the values of block next
    auto products = [&](auto with_values, const int next) {
        constexpr bool VALUES = decltype(with_values)::value;
        const unsigned char *kb = lds + slot(next + 1) * kRingBlock, *vb = lds + slot(next) * kRingBlock + 8192;
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int r = 0; r < V; ++r) x[ct][r / AL][r % AL] = 0.0f;
        // (one read behind the MFMAs that it serves: held up by a burst of them, the wave would issue no MFMA)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
#pragma unroll
            for (int ct = 0; ct < CT; ++ct) x[ct][FINE ? i & 1 : 0] = prefill_mfma(kf[i].v, qf[ct][FINE ? i >> 1 : i].v, x[ct][FINE ? i & 1 : 0]);
            kf[i].q = *(const u32x4 *)(kb + key_at(i));
            __builtin_amdgcn_sched_group_barrier(0x008, CT, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if constexpr (VALUES)
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) o[ct][FINE ? i : i & 3] = prefill_mfma(vf[i].v, pf[FINE ? ct : i >> 2].v, o[ct][FINE ? i : i & 3]);
            vf[i].q = *(const u32x4 *)(vb + value_at(i));
            if constexpr (VALUES) __builtin_amdgcn_sched_group_barrier(0x008, CT, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
    };
    // every wave has read its queries, and the first two blocks are in
    if constexpr (INT8) {
        stash(0);
        if (nblk > 1) {
            fetch(1);
            stash(1);
        }
        if (nblk > 2) fetch(2);
    }
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if constexpr (!INT8) request(2);
#pragma unroll
    for (int i = 0; i < 8; ++i) kf[i].q = *(const u32x4 *)(lds + key_at(i));
    __builtin_amdgcn_sched_barrier(0);
    products(std::false_type {}, 0);
    // Where the loop begins in the 32 bytes that are fetched at a time is worth 6 % (512 tokens behind 8000, by the number of 4-byte steps behind a border: 156,
    // 150, 150, 146, 148, 152, 154, 152 us; 4 x 2000 tokens 144 to 146.5, 2 x 1000 with 16 / 4 heads 23.9 to 24.9; FINE 154, 161, 172, 163, 160, 172, 154, 155, INT8 at 0, 2, 4, 6
    // steps 293, 306, 305, 294), so it is said.  (As the compiler of ROCm 7.2 lays out the code in front of it.)
    if constexpr (INT8 && FINE) asm volatile(".p2align 5\n\ts_nop 0\n\ts_nop 0\n\ts_nop 0\n\ts_nop 0\n\ts_nop 0\n\ts_nop 0");
    else if constexpr (!INT8 && FINE) asm volatile(".p2align 5");
    else if constexpr (!INT8) asm volatile(".p2align 5\n\ts_nop 0\n\ts_nop 0\n\ts_nop 0");
    for (int blk = 0; blk < nblk; ++blk) {
        // the block asked for goes where block blk - 1 was, which every wave has read for the last time in front of the barrier behind block blk - 1's softmax
        // (INT8: as much holds for block blk + 2, which is a register set ahead instead)
        if constexpr (INT8) {
            if (blk + 2 < nblk) stash(blk + 2);
            if (blk + 3 < nblk) fetch(blk + 3);
            if (blk < wave_nblk) softmax(blk);
        } else {
            request(blk + kLook);
            if (blk < wave_nblk) softmax(blk);
        }
        // block blk + 2 is in: everything but the requests just made
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (INT8) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        else asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)\n\ts_barrier" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_setprio(1);
        if (blk < wave_nblk) products(std::true_type {}, blk + 1);
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory"); // the requests past the end have landed

    float inv[CT];
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        float l = FINE ? l_run[ct] + swap16(l_run[ct]) : l_run[0] + l_run[1];
        l += swap32(l);
        inv[ct] = (INT8 ? vref : 1.0f) / l;
    }
    const size_t base = ((size_t)b * p.S + cs) * p.oStride + (size_t)(kvh * p.G + cj) * D;
    if (p.out_dtype == XFTHIP_BF16 && (((uintptr_t)p.out | ((size_t)p.oStride * 2)) & 15) == 0) {
        // whole rows through LDS, four of 256 bytes a store (from the registers: 16 stores of 32 rows' 16 bytes)
        __syncthreads(); // every wave's requests have landed, and its last operands are read
        constexpr int PITCH = 272;
        unsigned char *patch = lds + wave * (32 * PITCH);
#pragma unroll
        for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                for (int q = 0; q < AL / 4; ++q)
                    *(uint2 *)(patch + (TW * ct + tl) * PITCH + 256 / DT * dt + 16 * q + 8 * part) =
                            make_uint2(f32x2_to_bf16(o[ct][dt][4 * q] * inv[ct], o[ct][dt][4 * q + 1] * inv[ct]), f32x2_to_bf16(o[ct][dt][4 * q + 2] * inv[ct], o[ct][dt][4 * q + 3] * inv[ct]));
        const uint64_t orow = (uint64_t)(uintptr_t)((uint16_t *)p.out + base);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int r = 4 * i + (lane >> 4);
            const uint64_t dst = of_column(orow, r) + (lane & 15) * 16;
            const u32x4 w = *(const u32x4 *)(patch + r * PITCH + (lane & 15) * 16);
            if (c0 + r < ncols) *(u32x4 *)(uintptr_t)dst = w;
        }
        return;
    }
#pragma unroll
    for (int ct = 0; ct < CT; ++ct) {
        const size_t at_column = FINE ? of_column(base, TW * ct + tl) : base;
        if (limit[ct] > 0) store_direct<Acc, DT>(p, at_column, part, o[ct], inv[ct]);
    }
}

} // namespace xfthip
