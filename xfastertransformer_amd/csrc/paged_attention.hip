// Attention over a block-paged BF16 KV cache, the data path of xft::invokeAttention
// (reference src/kernels/attention_kernels.cpp:24-157, include/layers_attention.h:22-59).
//
// Cache layout (the caller's, part of that interface): [block_num][block_size][kv_heads][head_size]
// bf16; token t of a sequence lives in block block_table[t / block_size] at row t % block_size; a
// "slot" is block * block_size + row.
//
// Decode (one new token per sequence), as crossAttention does per (sequence, head): the new key and
// value rows go to their slots first, then scores = q . K^T in fp32 over context + 1 tokens,
// softmax(scale * scores) in fp32, out = P . V in fp32, narrowed to bf16.  HBM-bound: the query heads
// that share a key / value head are the columns of matrix products (paged_decode_kernel), so that the
// cache is read once a group; long contexts are split over workgroups whose partials a second kernel
// merges in a fixed order.
// Where this build departs from the reference's text: sequence b uses query / key / value row b
// (the reference reads row 0 for every sequence: no batch offset at attention_kernels.cpp:51,61,
// right only for batch_size = 1) and query head i uses KV head i / (q_heads / kv_heads) (the
// reference indexes the KV head with the query head, right only without grouped heads).
//
// Prefill: causal self-attention of every sequence over its own new tokens (the reference's
// selfAttention call), through this library's FP16-cache attention kernels on a scratch copy of the
// keys and values, and every token's key / value row stored to its slot (slot_mapping holds one entry
// per token; the reference's closures, marked "TODO: debug and fix", pass only slot_mapping[b]).
// All sequences of a call go through the same launches.
#include <algorithm>
#include <vector>

#include "attention_dev.h"
#include "attention_prefill.h"

namespace xfthip {
namespace {

struct PagedParams {
    uint16_t *out; // bf16 [batch, o_stride]
    const uint16_t *q; // bf16 [batch, q_stride]
    const uint16_t *kc, *vc; // paged caches
    const int *tables; // [batch, table_stride]
    const int *ctx; // tokens already cached per sequence (the new one excluded)
    float *part; // [batch, q_heads, nsplit, 130]: max, sum, out[128]
    int q_heads, kv_heads, q_stride, o_stride, table_stride, block_size, block_num, nsplit;
    float scale;
};

// rows of the new tokens -> their slots (keys and values), one workgroup per token
__global__ __launch_bounds__(256) void paged_store_kernel(uint16_t *kc, uint16_t *vc, const uint16_t *k, const uint16_t *v,
        const int *slots, int kv_stride, int row_elems, int slot_num) {
    const int tok = blockIdx.x;
    const int slot = slots[tok];
    if (slot < 0 || slot >= slot_num) return; // a slot outside the cache is dropped, never written
    const size_t dst = (size_t)slot * row_elems;
    const uint16_t *ks = k + (size_t)tok * kv_stride, *vs = v + (size_t)tok * kv_stride;
    for (int i = threadIdx.x * 8; i < row_elems; i += blockDim.x * 8) {
        *(u32x4 *)(kc + dst + i) = *(const u32x4 *)(ks + i);
        *(u32x4 *)(vc + dst + i) = *(const u32x4 *)(vs + i);
    }
}

union BFrag {
    bf16x8 v;
    uint32_t u[4];
    u32x4 q;
};

// grid (nsplit, kv_heads * column groups, batch), 256 threads.  head_size = 128.
// The columns of a workgroup are up to 16 query heads of one key / value head; a wave takes every fourth 32-token block of
// the workgroup's part of the context.
//   S^T[token][col] = K . Q^T: v_mfma_f32_16x16x32_bf16, A = key rows straight from the cache (products of bf16 values
//     in fp32, as before), lane (cl, g) holds dims 32 s + 8 g .. + 7 of token row cl in step s
//   O^T[dim][col] += V^T . P^T: the A operand wants 8 tokens of one dim a lane.  A lane loads dims 8 cl .. + 7 of 8 tokens
//     (whole 256-byte rows across 16 lanes), turns its 8 x 8 values round with 32 byte permutes and so holds the operands
//     of 8 products whose row r stands for dim 8 r + j - no LDS, no exchange.  Lane group g takes the tokens 4 g .. + 3 of
//     both 16-token score tiles, the ones whose probabilities it holds.
// The probabilities stay fp32: each goes in as the sum of three bf16 values (8 bits each, cut off one after the other), one
// product each.  Two parts were off by up to 2^-17, more than the exponential; the third costs 0.6 % of the call below, 4 % of one
// sequence of 64000 tokens.
// The next block's keys are requested once this block's scores are done, its values once this block's are turned; the
// cache rows of the block after that (a table look-up a lane) a block earlier.
// Bound by the cache's trip from HBM.  32 sequences of 2100 .. 4100 tokens, 32 query / 8 KV heads, 408 MB:
// 87 us, 4.7 TB/s (244 us with a workgroup a query head on the vector ALUs, every head of a group reading the cache again).  about 215
// registers, two workgroups a CU; held to three, 63 of them spill.
__global__ __launch_bounds__(256, 2) void paged_decode_kernel(PagedParams p) {
    constexpr int D = 128;
    __shared__ float s_m[4][16], s_l[4][16], s_o[4][16][D + 4];
    const int split = blockIdx.x, b = blockIdx.z;
    const int kvh = blockIdx.y % p.kv_heads, cg = blockIdx.y / p.kv_heads;
    const int G = p.q_heads / p.kv_heads, cols = min(16, G - cg * 16);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, cl = lane & 15;
    // tokens to attend to, the new one included (never more than the table describes)
    const int n = min(max(p.ctx[b], 0) + 1, p.table_stride * p.block_size);
    const int nblk = (n + 31) >> 5;
    const int b0 = (int)((long)nblk * split / p.nsplit), b1 = (int)((long)nblk * (split + 1) / p.nsplit);
    const int *table = p.tables + (size_t)b * p.table_stride;
    const size_t row_bytes = (size_t)p.kv_heads * D * 2;
    const char *kbase = (const char *)p.kc + kvh * (D * 2) + g * 16;
    const char *vbase = (const char *)p.vc + kvh * (D * 2) + cl * 16;

    // cache row of token 32 blk + (lane & 31); past the end the last token's (a valid row, masked below)
    auto row_of = [&](int blk) {
        const int t = min(32 * blk + (lane & 31), n - 1);
        const int at = t / p.block_size;
        return min(max(table[at], 0), p.block_num - 1) * p.block_size + (t - at * p.block_size); // a bad table entry reads a valid block
    };
    BFrag kf[2][4], vf[8], qf[4];
    auto load_keys = [&](int rows) {
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            const char *src = kbase + (size_t)__shfl(rows, 16 * a + cl, 64) * row_bytes;
#pragma unroll
            for (int s = 0; s < 4; ++s) kf[a][s].q = *(const u32x4 *)(src + 64 * s);
        }
    };
    auto load_values = [&](int rows) {
#pragma unroll
        for (int i = 0; i < 8; ++i) vf[i].q = *(const u32x4 *)(vbase + (size_t)__shfl(rows, 16 * (i >> 2) + 4 * g + (i & 3), 64) * row_bytes);
    };
    int blk = b0 + wave;
    int rows_next = 0;
    if (blk < b1) {
        const int rows = row_of(blk);
        load_keys(rows);
        load_values(rows);
        rows_next = row_of(min(blk + 4, nblk - 1));
    }
    {
        const uint16_t *qrow = p.q + (size_t)b * p.q_stride + (size_t)(kvh * G + cg * 16 + min(cl, cols - 1)) * D + 8 * g;
#pragma unroll
        for (int s = 0; s < 4; ++s) qf[s].q = *(const u32x4 *)(qrow + 32 * s);
    }
    float m = -INFINITY, l = 0.0f;
    f32x4 o[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = f32x4 {0.f, 0.f, 0.f, 0.f};
    for (; blk < b1; blk += 4) {
        const bool more = blk + 4 < b1; // (uniform over the wave)
        f32x4 sc[2];
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            sc[a] = f32x4 {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 4; ++s) sc[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[a][s].v, qf[s].v, sc[a], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (more) load_keys(rows_next);
        __builtin_amdgcn_sched_barrier(0);
        // ---- online softmax: this lane's column, tokens 16 a + 4 g + r of the block ----
        float bmax = -INFINITY;
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const bool seen = 32 * blk + 16 * a + 4 * g + r < n;
                sc[a][r] = seen ? sc[a][r] * p.scale : -INFINITY;
                bmax = fmaxf(bmax, sc[a][r]);
            }
        bmax = fmaxf(bmax, __shfl_xor(bmax, 16, 64));
        bmax = fmaxf(bmax, __shfl_xor(bmax, 32, 64));
        const float m_new = fmaxf(m, bmax);
        const float ref = m_new == -INFINITY ? 0.0f : m_new; // (nothing but minus infinity so far: exp() gives zeros)
        const float alpha = __expf(m - ref);
        m = m_new;
        float e[8], psum = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            e[i] = __expf(sc[i >> 2][i & 3] - ref);
            psum += e[i];
        }
        l = l * alpha + psum;
        BFrag pp[3];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            float x = e[2 * i], y = e[2 * i + 1];
#pragma unroll
            for (int part = 0; part < 3; ++part) {
                pp[part].u[i] = __builtin_amdgcn_perm(f2u(y), f2u(x), 0x07060302u);
                x -= u2f(f2u(x) & 0xFFFF0000u), y -= u2f(f2u(y) & 0xFFFF0000u);
            }
        }
        // ---- values: 8 tokens x 8 dims turned round, then O^T ----
        BFrag vt[8];
#pragma unroll
        for (int j = 0; j < 8; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                vt[j].u[i] = __builtin_amdgcn_perm(vf[2 * i + 1].u[j >> 1], vf[2 * i].u[j >> 1], (j & 1) ? 0x07060302u : 0x05040100u);
        __builtin_amdgcn_sched_barrier(0);
        if (more) {
            load_values(rows_next);
            rows_next = row_of(min(blk + 8, nblk - 1));
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            o[j] = o[j] * alpha;
#pragma unroll
            for (int part = 2; part >= 0; --part) o[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vt[j].v, pp[part].v, o[j], 0, 0, 0);
        }
    }
    // ---- merge the four waves; row 4 g + r of product j is dim 8 (4 g + r) + j ----
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (g == 0) s_m[wave][cl] = m, s_l[wave][cl] = l;
    bool nan = false;
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) nan |= o[j][r] != o[j][r];
    if (__builtin_amdgcn_ballot_w64(nan) == 0) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            float *dst = &s_o[wave][cl][8 * (4 * g + r)];
            *(f32x4 *)dst = f32x4 {o[0][r], o[1][r], o[2][r], o[3][r]};
            *(f32x4 *)(dst + 4) = f32x4 {o[4][r], o[5][r], o[6][r], o[7][r]};
        }
    } else {
        // A value that is not finite, times a part of a probability that is zero or times the zero of a slot past the end: the wave's blocks
        // again, a column at a time, one product a value in fp32 and none for those slots
        const float ref = m == -INFINITY ? 0.0f : m;
        for (int col = 0; col < cols; ++col) {
            float acc[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) acc[j] = 0.0f;
            for (blk = b0 + wave; blk < b1; blk += 4) {
                const int rows = row_of(blk);
                load_keys(rows);
                load_values(rows);
#pragma unroll
                for (int a = 0; a < 2; ++a) {
                    f32x4 sc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int s = 0; s < 4; ++s) sc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[a][s].v, qf[s].v, sc, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float e = __shfl(__expf(sc[r] * p.scale - ref), 16 * g + col, 64);
                        const bool seen = 32 * blk + 16 * a + 4 * g + r < n;
#pragma unroll
                        for (int j = 0; j < 8; ++j) {
                            const uint32_t w = vf[4 * a + r].u[j >> 1];
                            acc[j] = seen ? fmaf(e, u2f(j & 1 ? w & 0xFFFF0000u : w << 16), acc[j]) : acc[j];
                        }
                    }
                }
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                acc[j] += __shfl_xor(acc[j], 16, 64);
                acc[j] += __shfl_xor(acc[j], 32, 64);
                if (g == 0) s_o[wave][col][8 * cl + j] = acc[j];
            }
        }
    }
    __syncthreads();
    for (int v = threadIdx.x; v < cols * D; v += 256) {
        const int col = v / D, d = v % D, hq = kvh * G + cg * 16 + col;
        const float mm = fmaxf(fmaxf(s_m[0][col], s_m[1][col]), fmaxf(s_m[2][col], s_m[3][col]));
        float ll = 0.0f, acc = 0.0f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float f = s_m[w][col] == -INFINITY ? 0.0f : __expf(s_m[w][col] - mm);
            ll = fmaf(s_l[w][col], f, ll);
            acc = fmaf(s_o[w][col][d], f, acc);
        }
        if (!p.part) {
            p.out[(size_t)b * p.o_stride + hq * D + d] = f32_to_bf16_ref(acc / ll);
        } else {
            float *dst = p.part + (((size_t)b * p.q_heads + hq) * p.nsplit + split) * (D + 2);
            if (d == 0) dst[0] = mm, dst[1] = ll;
            dst[2 + d] = acc;
        }
    }
}

// grid (q_heads, batch), 128 threads: fixed-order merge of at most 32 splits, normalisation, bf16 output.  All the partials a
// thread needs are requested together: one round trip whatever the number of splits.
constexpr int kMaxSplits = 32;
__global__ __launch_bounds__(128) void paged_merge_kernel(PagedParams p) {
    constexpr int D = 128;
    __shared__ float s_m[kMaxSplits], s_l[kMaxSplits];
    const int hq = blockIdx.x, b = blockIdx.y, d = threadIdx.x;
    const float *src = p.part + ((size_t)b * p.q_heads + hq) * p.nsplit * (D + 2);
    if (d < p.nsplit) {
        const float2 ml = *(const float2 *)(src + (size_t)d * (D + 2));
        s_m[d] = ml.x, s_l[d] = ml.y;
    }
    float acc = 0.0f, ll = 0.0f, mm = -INFINITY;
    float t[kMaxSplits];
#pragma unroll
    for (int s = 0; s < kMaxSplits; ++s) t[s] = s < p.nsplit ? src[(size_t)s * (D + 2) + 2 + d] : 0.0f;
    __syncthreads();
    for (int s = 0; s < p.nsplit; ++s) mm = fmaxf(mm, s_m[s]);
#pragma unroll
    for (int s = 0; s < kMaxSplits; ++s)
        if (s < p.nsplit) {
            const float f = s_m[s] == -INFINITY ? 0.0f : __expf(s_m[s] - mm);
            ll = fmaf(s_l[s], f, ll);
            acc = fmaf(t[s], f, acc);
        }
    p.out[(size_t)b * p.o_stride + hq * D + d] = f32_to_bf16_ref(acc / ll);
}

// ---- prefill: the sequences of a call side by side ---------------------------------------------------------------
// Sequence i of a launch: tokens from row row0[i] on, rows[i] of them, 32-token blocks from blk0[i] on in the scratch copy (which holds blk0[n]
// blocks a head).  An attention kernel takes the sequences first .. first + many - 1; grp0: workgroups of an XCD in front of the k-th part
// of the walk over their (sequence, KV head) pairs; scaled: how many of them take queries with the scale's power of two.  By value: no copy in front of the launch.
constexpr int kSeqs = 64, kGroups = 256;
struct SeqBatch {
    int n, first, many, scaled;
    int row0[kSeqs], rows[kSeqs], blk0[kSeqs + 1];
    int grp0[kGroups + 1];
    PrefillBands bands;
};

__device__ inline int seq_of_block(const SeqBatch &s, int blk) {
    int lo = 0, hi = s.n - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (s.blk0[mid] <= blk) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// One workgroup a (KV head, 32-token block): a token's key and value row go to its slot as they are, to the scratch copy in FP16,
// the values turned into the [dim][32 slots] tile the attention kernels read (kvcache.h).  Slots of a block past the sequence's
// end are zero: what lies there is multiplied by a probability of zero.
// (6 sequences of 750 .. 1500 tokens, 32 query / 8 KV heads: the slots' store, a fused q | k | v copy, an append and an attention launch a
// sequence took 11 + 28 + 6 x (14 + 43) us, 366 the call; one store and one attention launch 143.  3 x 60 tokens 38 -> 13 us.)
__global__ __launch_bounds__(256) void paged_prefill_store_kernel(SeqBatch s, KvView kv, uint16_t *kc, uint16_t *vc, const uint16_t *k, const uint16_t *v,
        const int *slots, int kv_stride, int slot_num) {
    __shared__ __attribute__((aligned(16))) uint16_t tile[128 * 32];
    const int kvh = blockIdx.y, blk = blockIdx.x, i = seq_of_block(s, blk);
    const int t0 = 32 * (blk - s.blk0[i]), tl = threadIdx.x >> 3, c = threadIdx.x & 7;
    const bool live = t0 + tl < s.rows[i];
    const size_t tok = (size_t)s.row0[i] + t0 + tl;
    u32x4 x[4]; // keys 8 c .. and 64 + 8 c .., values the same
#pragma unroll
    for (int e = 0; e < 4; ++e) x[e] = u32x4 {0u, 0u, 0u, 0u};
    if (live) {
        const uint16_t *kr = k + tok * kv_stride + kvh * 128 + 8 * c, *vr = v + tok * kv_stride + kvh * 128 + 8 * c;
        x[0] = *(const u32x4 *)kr, x[1] = *(const u32x4 *)(kr + 64), x[2] = *(const u32x4 *)vr, x[3] = *(const u32x4 *)(vr + 64);
        const int slot = slots[tok];
        if (slot >= 0 && slot < slot_num) { // a slot outside the cache is dropped, never written
            const size_t dst = ((size_t)slot * kv.H + kvh) * 128 + 8 * c;
            *(u32x4 *)(kc + dst) = x[0], *(u32x4 *)(kc + dst + 64) = x[1];
            *(u32x4 *)(vc + dst) = x[2], *(u32x4 *)(vc + dst + 64) = x[3];
        }
    }
    uint16_t h[4][8];
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int j = 0; j < 8; ++j) h[e][j] = f32_to_fp16_bits(u2f(j & 1 ? x[e][j >> 1] & 0xFFFF0000u : x[e][j >> 1] << 16));
    uint16_t *kd = (uint16_t *)kv.k + ((size_t)kvh * kv.S + 32 * blk + tl) * 128 + 8 * c;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        u32x4 w;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = (uint32_t)h[e][2 * j] | ((uint32_t)h[e][2 * j + 1] << 16);
        *(u32x4 *)(kd + 64 * e) = w;
    }
    const int slot_in = v_slot(tl);
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int j = 0; j < 8; ++j) tile[(64 * e + 8 * c + j) * 32 + slot_in] = h[2 + e][j];
    __syncthreads();
    u32x4 *vd = (u32x4 *)((uint16_t *)kv.v + ((size_t)kvh * (kv.S / 32) + blk) * 128 * 32);
#pragma unroll
    for (int e = 0; e < 2; ++e) vd[threadIdx.x + 256 * e] = ((const u32x4 *)tile)[threadIdx.x + 256 * e];
}

// the parameters of sequence i of a batch
__device__ inline AttnParams seq_params(const AttnParams &all, const SeqBatch &s, int i) {
    AttnParams p = all;
    p.S = s.rows[i];
    p.CG = (p.S * p.G + 15) / 16;
    p.q += (size_t)s.row0[i] * p.qStride;
    p.out = (uint16_t *)p.out + (size_t)s.row0[i] * p.oStride;
    p.kv.k = (uint16_t *)p.kv.k + (size_t)s.blk0[i] * 32 * 128;
    p.kv.v = (uint16_t *)p.kv.v + (size_t)s.blk0[i] * 32 * 128;
    return p;
}

// attn_prefill32_kernel over sequences, the longest first.  Group k of 8 pairs has n(k) column groups, those of its longest sequence.  An XCD walks a band in levels,
// from the longest walk down: levels n(k) - 1 .. n(k + 1), which groups k and those in front of it in its band reach, are part k.
// (6 sequences of 750 .. 1500 tokens, 32 query / 8 KV heads: group after group 113 us the call, so 106; 7 of 600 .. 1200, 16 / 4 heads 58 and 52)
template <bool FINE>
__global__ __launch_bounds__(256, 2) void paged_prefill_attn_kernel(AttnParams all, SeqBatch s) {
    __shared__ __attribute__((aligned(16))) unsigned char lds[kRingLds];
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    int group = 0, hi = (s.many * all.kv.H + 7) / 8 - 1;
    while (group < hi) {
        const int mid = (group + hi + 1) >> 1;
        if (s.grp0[mid] <= slot) group = mid;
        else hi = mid - 1;
    }
    int first, width;
    prefill_band(s.bands, group, first, width);
    const int reach = group - first + 1, at = slot - s.grp0[group];
    const int level = (s.rows[group * 8 / all.kv.H] * all.G + 127) / 128 - 1 - at / reach;
    const int pair = (first + at % reach) * 8 + xcd, i = pair / all.kv.H;
    if (i >= s.many) return;
    const AttnParams p = seq_params(all, s, s.first + i);
    const int ncg = (p.S * p.G + 127) / 128;
    if (level >= ncg) return; // (a longer sequence shares the group)
    attn_prefill_ring_unit<false, FINE>(p, pair % all.kv.H, level, 0, lds, i >= s.scaled);
}

// attn_kernel over sequences, each walked by one workgroup a column group: grid (KV heads x the longest's column groups, sequences)
__global__ __launch_bounds__(256, 3) void paged_prefill_few_kernel(AttnParams all, SeqBatch s) {
    __shared__ AttnLds<4> lds;
    const AttnParams p = seq_params(all, s, s.first + blockIdx.y);
    const int cg = blockIdx.x / all.kv.H;
    if (cg >= p.CG) return;
    attn_unit<false, 4, false>(p, 0, blockIdx.x % all.kv.H, cg, 0, lds, [] { __syncthreads(); });
}

// Rows of `out` and of `x` (strides and widths in elements) that lie such that writing one row of the former may change another row, or another
// head, of the latter: a workgroup that writes its results must not do so before all others have read.
bool in_the_way(const void *out, long o_stride, long o_width, const void *x, long x_stride, long x_width, long rows) {
    const long d = ((const char *)out - (const char *)x) / 2;
    if (d >= (rows - 1) * x_stride + x_width || -d >= (rows - 1) * o_stride + o_width) return false;
    if (o_stride != x_stride) return true;
    const long at = (d % x_stride + x_stride) % x_stride; // where a row of `out` begins beside the rows of `x`
    return d != 0 && (at < x_width || x_stride - at < o_width);
}

// rows of 16-byte pieces -> contiguous rows
__global__ __launch_bounds__(256) void paged_copy_rows_kernel(uint16_t *dst, const uint16_t *src, int stride, int width) {
    for (int i = threadIdx.x * 8; i < width; i += blockDim.x * 8) *(u32x4 *)(dst + (size_t)blockIdx.x * width + i) = *(const u32x4 *)(src + (size_t)blockIdx.x * stride + i);
}

int check_common(const void *out, const void *q, const void *k, const void *v, int q_heads, int kv_heads, int head_size, int q_stride,
        int kv_stride, int o_stride, const void *kc, const void *vc, int block_size) {
    XFT_REQUIRE(out && q && k && v && kc && vc, "xfthip_paged_attention: null argument");
    XFT_REQUIRE(head_size == 128, "xfthip_paged_attention: head size %d unsupported (128 only)", head_size);
    XFT_REQUIRE(q_heads > 0 && kv_heads > 0 && q_heads % kv_heads == 0, "xfthip_paged_attention: bad head counts %d / %d", q_heads, kv_heads);
    XFT_REQUIRE(block_size > 0, "xfthip_paged_attention: bad block size");
    XFT_REQUIRE(q_stride >= q_heads * 128 && kv_stride >= kv_heads * 128 && o_stride >= q_heads * 128, "xfthip_paged_attention: stride too small");
    XFT_REQUIRE(q_stride % 8 == 0 && kv_stride % 8 == 0, "xfthip_paged_attention: strides must be multiples of 8 elements");
    XFT_REQUIRE((((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)kc | (uintptr_t)vc) & 15) == 0,
            "xfthip_paged_attention: q, k, v and the caches must be 16-byte aligned");
    return 0;
}

// Which form takes the sequences of a launch, the longest first: the first `many` that for many columns, `scaled` of them with queries that carry the scale's power of two
struct SeqForms {
    int scaled, many;
    bool fine;
};
SeqForms seq_forms(const int *rows, int n, int G, int kv_heads) {
    SeqForms f = {0, 0, false};
    const long enough = 4L * device_cu_count();
    long waves = 0; // of 16 columns, of those that attention_launch would not take to the form for many columns
    for (int i = 0; i < n; ++i) {
        const long w = (long)kv_heads * (((long)rows[i] * G + 15) / 16);
        if (rows[i] > 1 && w >= enough) ++f.scaled;
        else waves += w;
    }
    // Those that it would, and the others with them where they are enough together (12 x 200 tokens, 32 query / 8 KV heads 21 us against 52 in the form for few columns, 8 x 600,
    // 16 / 4 heads 29 against 79), with their queries as they are, as the form that each would take alone has them
    f.many = waves >= enough ? n : f.scaled;
    long groups = 0, walks = 0; // column groups of a KV head, the tokens that their columns see on average
    for (int i = 0; i < f.many; ++i) {
        const long g = ((long)rows[i] * G + 127) / 128;
        groups += g, walks += g * (rows[i] / 2);
    }
    // (Blocks a CU in brackets, 32 / 8 heads, us of the call in 32 x 32 and in 16 x 16 MFMAs: 6 sequences of 750 to 1500 tokens (120) 98.0 and 94.5, 3000 and 30 of 60 (135) 103.9 and 102.6, 1700, 1103, 701 (71)
    // 71.0 and 68.9, 2 of 2500, 16 / 4 heads (96) 82.2 and 81.1, 4 of 900 (51) 51.1 and 50.8; but 1700 and 2 of 200 (45) 72.6 and 74.2, 1500 and 60 of 60 (37) 61.2 and 62.6, 1200 and 63 of 64 (26) 47.6 and
    // 48.6.  By the longest sequence's walk the last two would be 120 and 92.)
    f.fine = f.many > 0 && prefill_fine(false, groups * kv_heads, walks / groups, 50);
    return f;
}
// sequences of a launch: at most kSeqs, and kGroups groups of 8 (sequence, KV head) pairs
int seqs_per_launch(int kv_heads) { return std::max(1, std::min(kSeqs, kGroups * 8 / kv_heads - 1)); }

} // namespace
} // namespace xfthip

using namespace xfthip;

extern "C" int xfthip_paged_attention_decode(void *out, const void *q, const void *k, const void *v, int q_heads, int kv_heads,
        int head_size, int q_stride, int kv_stride, int o_stride, float scale, int batch, void *kcache, void *vcache, int block_num,
        int block_size, const int *block_tables, int table_stride, const int *context_lens, const int *slot_mapping,
        int max_context, xfthip_stream_t stream) {
    if (int rc = check_common(out, q, k, v, q_heads, kv_heads, head_size, q_stride, kv_stride, o_stride, kcache, vcache, block_size)) return rc;
    XFT_REQUIRE(batch > 0 && block_tables && context_lens && slot_mapping && table_stride > 0, "xfthip_paged_attention_decode: bad argument");
    XFT_REQUIRE(max_context >= 0 && (long)(max_context / block_size + 1) <= (long)table_stride,
            "xfthip_paged_attention_decode: a context of %d + 1 tokens needs %d table entries a sequence, the table has %d", max_context,
            max_context / block_size + 1, table_stride);
    XFT_REQUIRE(block_num > 0, "xfthip_paged_attention_decode: bad block count");
    hipStream_t st = (hipStream_t)stream;
    // About one workgroup a CU, at least one 32-token block a wave (1, 2 or 4 workgroups a CU: 1 x 1000 tokens, 8 KV heads 10.3 / 11.7 / 11.6 us,
    // 64 x 500, 4 KV heads 15.0 / 17.5 / 19.1, 1 x 9000 16.8 / 16.8 / 16.9, 32 x 4100 86.6 / 87.2 / 85.2), 32 splits at most: below 8 (sequence, KV head,
    // column group) units part of the CUs stay idle (64 splits cost 1 x 9000 2.5 us; with 32, 1 x 32000 tokens, 8 query / 1 KV heads take 25 us, 1 x 100000 54,
    // against 49 and 79 with a workgroup a query head and 64 splits)
    const int colgroups = (q_heads / kv_heads + 15) / 16, units = batch * kv_heads * colgroups;
    int nsplit = (device_cu_count() + units - 1) / units;
    const int cap = (max_context + 1 + 127) / 128;
    if (nsplit > cap) nsplit = cap;
    if (nsplit > kMaxSplits) nsplit = kMaxSplits;
    if (nsplit < 1) nsplit = 1;
    // The parts of any split call: below 2 CUs workgroups of 16 columns (4.3 MB on 256 CUs).  Taken by the stream's first call, split or not, so that
    // none behind it allocates (a captured one must not).  Results that may lie over queries still to be read go by way of it as well.
    const bool apart = !in_the_way(out, o_stride, q_heads * 128, q, q_stride, q_heads * 128, batch);
    const size_t any = (size_t)2 * device_cu_count() * 16 * 130, need = (size_t)batch * q_heads * nsplit * 130;
    void *part = nullptr;
    if (int rc = stream_scratch(kScratchPagedParts, st, std::max(any, apart ? 0 : need) * sizeof(float), false, &part)) return rc;
    if (nsplit == 1 && apart) part = nullptr;
    PagedParams p = {};
    p.out = (uint16_t *)out, p.q = (const uint16_t *)q, p.kc = (const uint16_t *)kcache, p.vc = (const uint16_t *)vcache;
    p.tables = block_tables, p.ctx = context_lens, p.part = (float *)part;
    p.q_heads = q_heads, p.kv_heads = kv_heads, p.q_stride = q_stride, p.o_stride = o_stride, p.table_stride = table_stride;
    p.block_size = block_size, p.block_num = block_num, p.nsplit = nsplit, p.scale = scale;
    hipLaunchKernelGGL(paged_store_kernel, dim3(batch), dim3(256), 0, st, (uint16_t *)kcache, (uint16_t *)vcache, (const uint16_t *)k,
            (const uint16_t *)v, slot_mapping, kv_stride, kv_heads * 128, block_num * block_size);
    hipLaunchKernelGGL(paged_decode_kernel, dim3(nsplit, kv_heads * colgroups, batch), dim3(256), 0, st, p);
    if (part) hipLaunchKernelGGL(paged_merge_kernel, dim3(q_heads, batch), dim3(128), 0, st, p);
    XFT_CHECK_HIP(hipGetLastError());
    return 0;
}

extern "C" int xfthip_attention_prefill_form(int cache_int8, int q_heads, int kv_heads, int batch, int tokens, int past, int *form) {
    XFT_REQUIRE(form && batch > 0 && tokens > 0 && past >= 0 && kv_heads > 0 && q_heads % kv_heads == 0, "xfthip_attention_prefill_form: bad argument");
    *form = attention_prefill_form(cache_int8 != 0, q_heads / kv_heads, (long)batch * kv_heads, tokens, past);
    return 0;
}

extern "C" int xfthip_paged_attention_prefill_forms(int q_heads, int kv_heads, int batch, const int *token_lens_host, int *forms) {
    XFT_REQUIRE(forms && token_lens_host && batch > 0 && kv_heads > 0 && q_heads % kv_heads == 0, "xfthip_paged_attention_prefill_forms: bad argument");
    std::vector<int> order(batch), rows;
    for (int b = 0; b < batch; ++b) {
        XFT_REQUIRE(token_lens_host[b] > 0, "xfthip_paged_attention_prefill_forms: sequence %d has %d tokens", b, token_lens_host[b]);
        order[b] = b;
    }
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return token_lens_host[x] > token_lens_host[y]; });
    const int G = q_heads / kv_heads, per_launch = seqs_per_launch(kv_heads);
    for (int b = 0; b < batch; b += per_launch) {
        const int n = std::min(per_launch, batch - b);
        rows.clear();
        for (int i = 0; i < n; ++i) rows.push_back(token_lens_host[order[b + i]]);
        const SeqForms f = seq_forms(rows.data(), n, G, kv_heads);
        for (int i = 0; i < n; ++i) forms[order[b + i]] = n == 1 ? attention_prefill_form(false, G, kv_heads, rows[0], 0) : i >= f.many ? 0 : f.fine ? 2 : 1;
    }
    return 0;
}

extern "C" int xfthip_paged_attention_prefill(void *out, const void *q, const void *k, const void *v, int q_heads, int kv_heads,
        int head_size, int q_stride, int kv_stride, int o_stride, float scale, int batch, const int *token_lens_host, void *kcache,
        void *vcache, int block_num, int block_size, const int *slot_mapping, xfthip_stream_t stream) {
    if (int rc = check_common(out, q, k, v, q_heads, kv_heads, head_size, q_stride, kv_stride, o_stride, kcache, vcache, block_size)) return rc;
    XFT_REQUIRE(batch > 0 && token_lens_host && slot_mapping && block_num > 0, "xfthip_paged_attention_prefill: bad argument");
    XFT_REQUIRE(o_stride % 8 == 0, "xfthip_paged_attention_prefill: o_stride must be a multiple of 8 elements");
    hipStream_t st = (hipStream_t)stream;
    for (int b = 0; b < batch; ++b)
        XFT_REQUIRE(token_lens_host[b] > 0, "xfthip_paged_attention_prefill: sequence %d has %d tokens", b, token_lens_host[b]);
    // launches of several sequences, the longest first
    const int per_launch = seqs_per_launch(kv_heads);
    std::vector<int> order(batch), first(batch);
    for (int b = 0, at = 0; b < batch; at += token_lens_host[b], ++b) order[b] = b, first[b] = at;
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return token_lens_host[x] > token_lens_host[y]; });
    // Scratch for the keys and values of any lengths that add up to these tokens (a sequence of a launch fills its last 32-token block), with the bytes of
    // the whole q | k | v rows: a later call of no more bytes allocates nothing, whatever its lengths (a captured one must not)
    size_t total = 0;
    for (int b = 0; b < batch; ++b) total += token_lens_host[b];
    const size_t kv_bytes = (total + 31 * kSeqs) * kv_heads * 128 * 4;
    const size_t q_bytes = total * q_heads * 128 * 2, copied = total * kv_heads * 128 * 2;
    // results that may lie over rows still to be read: those rows are read from a copy
    const bool q_apart = !in_the_way(out, o_stride, q_heads * 128, q, q_stride, q_heads * 128, (long)total);
    const bool kv_apart = batch <= per_launch || (!in_the_way(out, o_stride, q_heads * 128, k, kv_stride, kv_heads * 128, (long)total)
                                                         && !in_the_way(out, o_stride, q_heads * 128, v, kv_stride, kv_heads * 128, (long)total));
    void *scratch = nullptr;
    if (int rc = stream_scratch(kScratchPagedKv, st, kv_bytes + q_bytes + (kv_apart ? 0 : 2 * copied), false, &scratch)) return rc;
    auto copy_rows = [&](const void *&x, int &stride, int heads, size_t at) {
        uint16_t *to = (uint16_t *)((char *)scratch + at);
        hipLaunchKernelGGL(paged_copy_rows_kernel, dim3((unsigned)total), dim3(256), 0, st, to, (const uint16_t *)x, stride, heads * 128);
        x = to, stride = heads * 128;
    };
    if (!q_apart) copy_rows(q, q_stride, q_heads, kv_bytes);
    if (!kv_apart) {
        int stride = kv_stride;
        copy_rows(k, stride, kv_heads, kv_bytes + q_bytes);
        copy_rows(v, kv_stride, kv_heads, kv_bytes + q_bytes + copied);
    }
    const int G = q_heads / kv_heads;
    for (int b = 0; b < batch; ++b) // likewise what one of these sequences by itself splits its keys through
        if (attention_split_count(token_lens_host[b], kv_heads * ((token_lens_host[b] * G + 15) / 16)) > 1) {
            AttnWorkspace of_stream;
            if (int rc = attention_stream_workspace(st, &of_stream)) return rc;
            break;
        }
    for (int b = 0; b < batch; b += per_launch) {
        SeqBatch s = {};
        s.n = std::min(per_launch, batch - b);
        for (int i = 0; i < s.n; ++i) {
            const int S = token_lens_host[order[b + i]];
            s.row0[i] = first[order[b + i]], s.rows[i] = S, s.blk0[i + 1] = s.blk0[i] + (S + 31) / 32;
        }
        const int blocks = s.blk0[s.n];
        KvView kv = {};
        kv.B = 1, kv.H = kv_heads, kv.S = 32 * blocks, kv.D = 128;
        kv.k = scratch, kv.v = (uint16_t *)scratch + (size_t)32 * blocks * kv_heads * 128;
        hipLaunchKernelGGL(paged_prefill_store_kernel, dim3(blocks, kv_heads), dim3(256), 0, st, s, kv, (uint16_t *)kcache, (uint16_t *)vcache,
                (const uint16_t *)k, (const uint16_t *)v, slot_mapping, kv_stride, block_num * block_size);
        if (s.n == 1) {
            // one sequence: the rules of attention over a contiguous cache, splits of a short one's keys among them
            xfthip_kvcache cache = {};
            cache.kv = kv, cache.maxSeq = s.rows[0];
            XFT_CHECK_HIP(hipGetLastError());
            if (int rc = attention_launch(&cache, (const uint16_t *)q + (size_t)s.row0[0] * q_stride, q_stride,
                        (uint16_t *)out + (size_t)s.row0[0] * o_stride, o_stride, XFTHIP_BF16, 1, s.rows[0], q_heads, scale, 0, nullptr, 0, st, nullptr, false))
                return rc;
            continue;
        }
        AttnParams p = {};
        p.kv = kv, p.q = (const uint16_t *)q, p.qStride = q_stride, p.out = out, p.oStride = o_stride, p.out_dtype = XFTHIP_BF16;
        p.B = 1, p.G = G, p.scale = scale, p.nsplit = 1;
        const SeqForms forms = seq_forms(s.rows, s.n, G, kv_heads);
        s.first = 0, s.scaled = forms.scaled, s.many = forms.many;
        const int groups = (s.many * kv_heads + 7) / 8;
        s.bands = prefill_bands(groups);
        auto levels = [&](int g) { return (int)(((long)s.rows[g * 8 / kv_heads] * G + 127) / 128); }; // (the sequences are sorted: the group's first pair belongs to its longest)
        for (int g = 0; g < groups; ++g) {
            int band, width;
            prefill_band(s.bands, g, band, width);
            s.grp0[g + 1] = s.grp0[g] + (levels(g) - (g + 1 < band + width ? levels(g + 1) : 0)) * (g - band + 1);
        }
        if (s.many > 0 && forms.fine) hipLaunchKernelGGL(paged_prefill_attn_kernel<true>, dim3(8 * s.grp0[groups]), dim3(256), 0, st, p, s);
        else if (s.many > 0) hipLaunchKernelGGL(paged_prefill_attn_kernel<false>, dim3(8 * s.grp0[groups]), dim3(256), 0, st, p, s);
        s.first = s.many, s.many = s.n - s.many;
        if (s.many > 0)
            hipLaunchKernelGGL(paged_prefill_few_kernel, dim3(kv_heads * ((s.rows[s.first] * G + 15) / 16), s.many), dim3(256), 0, st, p, s);
        XFT_CHECK_HIP(hipGetLastError());
    }
    return 0;
}
