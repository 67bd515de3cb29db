// Dequant-fused weight-only GEMM for many activation rows (M > 32): the prefill shape.
// Replaces MMHelper::compute* (reference src/utils/matmul_helper.h:565-1705) at large M, where
// the reference switches to AMX (oneDNN) kernels.  The kernels live in qgemm_mfma_impl.h and
// qgemm_direct_impl.h; this file picks the weight kind and the tile.
#include <math.h>

#include <algorithm>
#include <mutex>

#include "qgemm.h"

namespace xfthip {

// weak: a library for models with BF16 weights only is built without the quantised kinds (build.py)
__attribute__((weak)) int qgemm_mfma_int8(const SkinnyParams &p, hipStream_t stream);
__attribute__((weak)) int qgemm_mfma_int8z(const SkinnyParams &p, hipStream_t stream);
__attribute__((weak)) int qgemm_mfma_uint4(const SkinnyParams &p, hipStream_t stream);
__attribute__((weak)) int qgemm_mfma_nf4(const SkinnyParams &p, hipStream_t stream);
int qgemm_mfma_bf16(const SkinnyParams &p, hipStream_t stream);

namespace {

__device__ inline float silu_split(float x) {
    return x / (1.0f + fast_exp(-x));
}

// One thread per VEC neighbouring output values of a row (4 where N allows 16-byte part loads, else 1): the K parts are
// added in order (the same result on every run), then the epilogue of the call.  p.C / p.ldc / p.c_dtype / p.epi are
// the caller's.
template <int VEC>
__global__ __launch_bounds__(256) void qgemm_split_finish_kernel(SkinnyParams p) {
    const int nv = p.N / VEC;
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (size_t)p.M * nv) return;
    const int m = (int)(idx / nv), n0 = (int)(idx - (size_t)m * nv) * VEC;
    int row_out = m;
    if (p.group) {
        // the parts hold the rows where C holds them; rows past the last weight's were never written
        int total = 0;
        for (int e = 0; e < p.group_n; ++e) total += p.rows_dev[e * p.rows_stride];
        if (m >= total) return;
    } else if (p.rows_dev) {
        if (m >= p.rows_dev[0]) return;
        row_out = m + p.rows_dev[2];
    }
    float x[VEC];
#pragma unroll
    for (int v = 0; v < VEC; ++v) x[v] = 0.0f;
    for (int s = 0; s < p.ksplit; ++s) {
        const float *src = p.split_part + ((size_t)s * p.M + m) * p.N + n0;
        if constexpr (VEC == 4) {
            const float4 t = *(const float4 *)src;
            x[0] += t.x, x[1] += t.y, x[2] += t.z, x[3] += t.w;
        } else {
            x[0] += src[0];
        }
    }
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
        const int n = n0 + v;
        float y = x[v];
        switch (p.epi) {
            case XFTHIP_EPI_BIAS: y += p.bias[n]; break;
            case XFTHIP_EPI_SILU: y = silu_split(y); break;
            case XFTHIP_EPI_GELU: {
                const float e = fast_exp(1.702f * y);
                y = e / (e + 1.0f) * y;
                break;
            }
            case XFTHIP_EPI_RESMUL: y *= load_as_f32(p.res, p.res_dtype, (size_t)m * p.ldres + n); break;
            case XFTHIP_EPI_RESIDENTIAL:
                if (p.bias) y += p.bias[n];
                y += load_as_f32(p.res, p.res_dtype, (size_t)m * p.ldres + n);
                break;
            case XFTHIP_EPI_RESEXT:
                if (p.bias) y += p.bias[n];
                y = fmaf(p.gamma, load_as_f32(p.res, p.res_dtype, (size_t)m * p.ldres + n), y);
                break;
            default: break;
        }
        x[v] = y;
    }
    const size_t ci = (size_t)row_out * p.ldc + n0;
    if constexpr (VEC == 4) {
        // whole 16-byte (fp32) or 8-byte (16-bit) stores where the row start allows them
        if (p.c_dtype == XFTHIP_F32 && ((((uintptr_t)p.C) | ((size_t)p.ldc * 4)) & 15) == 0) {
            *(float4 *)((float *)p.C + ci) = make_float4(x[0], x[1], x[2], x[3]);
            return;
        }
        if (p.c_dtype == XFTHIP_BF16 && ((((uintptr_t)p.C) | ((size_t)p.ldc * 2)) & 7) == 0) {
            const uint32_t lo = f32x2_to_bf16(x[0], x[1]);
            const uint32_t hi = f32x2_to_bf16(x[2], x[3]);
            *(uint2 *)((uint16_t *)p.C + ci) = make_uint2(lo, hi);
            return;
        }
    }
#pragma unroll
    for (int v = 0; v < VEC; ++v) store_from_f32(p.C, p.c_dtype, ci + v, x[v]);
}

// Which tile, how many parts of K and how many K groups a workgroup: the cheapest by a cost model of the launch.
//   time = start + rounds of resident blocks (steps of 64 k times what a step costs with so many blocks on a CU, + pipeline fill and
//          results) + the sum of the parts of a split K
// A CU's blocks are those of the XCD with the most (band_rows); a partly filled round costs between the blocks of the fullest CU and
// those of the average one, a partly filled device a little less a step than a full one.  The constants (microseconds) are a
// least-squares fit to 35000 timings on weights that do not fit the Infinity Cache: 340 shapes of 1024 .. 28672 columns x 1024 .. 14336 deep,
// 33 to 4096 rows, 1 to 8 parts, the five weight kinds, of the 96- and 128-row tiles on 32 x 32 x 16 MFMAs: 1.01 to 1.02 times the best form's time on average over those
// cells then (1.33 at worst).  On the kernels as they are, whose 128 x 128 tile gained the most, over 3200 to 4500 shapes a kind: INT8 1.023 on average, 1.12 for one in twenty, 1.65 at worst (87 x 22016 x 4096
// 50 us, best 30); UINT4 1.009, 1.06, 1.41 (1593 x 11264 x 2048 90, 64); NF4 1.015, 1.10, 1.23; BF16 1.038, 1.19, 1.55 (390 x 2048 x 2048 20.5, 13.2); their times come out 14 to 29 % too
// long (INT8).  In words: the largest tile that gives most CUs a block, K split or taken in two groups where that takes it to
// about a block a CU, and for few rows parts of K until there are two or three 32- or 64-row blocks a CU.  Against thresholds on the rows
// (which left 700 rows x 4096 columns on 64-row tiles and split 128 rows too little) and bands padded to 8 row blocks: INT8 1.15 times as
// fast in the geometric mean over the cells, with zero points 1.17, UINT4 1.12, NF4 1.19, BF16 1.43; 900 x 4096 x 14336 INT8 142 -> 113 us,
// 128 x 4096 x 14336 46 -> 34, 600 x 12288 x 4096 94 -> 65, 64 x 28672 x 4096 57 -> 33.
// Several weights behind one launch (the experts of a sparse MLP): the same, without K groups, over the row blocks to be expected.  Against
// 64-row tiles with K in up to 4 parts throughout: a Mixtral-8x7B layer, INT8, 400 tokens 549 -> 490 us, 1000 tokens 1060 -> 940; 8 experts
// of width 2816 at width 2048, BF16, 6132 tokens, two layers and all else 3.28 -> 2.98 ms.
// 96 x 256, for 65 .. 96 rows, experts with some more than 64 and counts that are one or a few more than a multiple of 128: its constants are those of 128 x 256 by the ratios of two
// fits to 100 timings each.  Products that take it, 1024 .. 57344 columns x 1024 .. 28672 deep, 33 .. 2800 rows, against the same without it: INT8 and BF16 0.89 of the time in the
// geometric mean (384 x 28672 x 4096 INT8 with SwiGLU 100 -> 87 us, 900 x 11008 x 4096 94 -> 82, 407 x 2560 x 22016 BF16 81 -> 56), UINT4 0.91, NF4 0.94; a Mixtral-8x7B layer, INT8, of 256 / 290 / 580 / 1024 tokens
// 381 / 425 / 640 / 873 -> 369 / 377 / 597 / 872 us, UINT4, 256 tokens 363 -> 336.
struct TileCost {
    int rows, cols, kgroups, resident;
    float fixed; // a block's pipeline fill and results
    float step[4], more[4]; // per step of a block alone on a CU; per further resident block.  INT8, BF16, NF4, UINT4
};
constexpr TileCost kTiles[] = {
        {32, 128, 1, 4, 0.6f, {0.26f, 0.0f, 0.39f, 0.247f}, {0.15f, 0.0f, 0.26f, 0.143f}},
        {64, 128, 1, 4, 1.2f, {0.35f, 0.56f, 0.51f, 0.357f}, {0.27f, 0.34f, 0.43f, 0.275f}},
        {128, 128, 1, 2, 1.7f, {0.71f, 0.64f, 0.90f, 0.71f}, {0.26f, 0.36f, 0.65f, 0.26f}},
        {128, 128, 2, 1, 4.3f, {1.0f, 1.14f, 1.38f, 1.0f}, {}},
        {96, 256, 1, 2, 2.3f, {0.80f, 0.85f, 1.25f, 0.75f}, {0.525f, 0.54f, 1.025f, 0.575f}},
        {128, 256, 1, 2, 3.1f, {0.92f, 0.93f, 1.59f, 0.92f}, {0.73f, 0.77f, 1.34f, 0.73f}},
        {128, 256, 2, 1, 8.7f, {1.49f, 1.8f, 2.63f, 1.49f}, {}},
};

// What 96 x 256 has to gain by the model before a product takes it: 700 products that the model alone gives to it, against what they take
// without it, lost more than 2 % in 12 % of cases (NF4 19) and up to 1.2 times (800 x 14336 x 28672 BF16 665 -> 755 us, 696 x 2560 x 11008 NF4 79 -> 91), mostly where the model saw
// little to gain.  With these prices 4 %, and 0.931 of the time in the geometric mean (0.928 without).  Left: 4 row blocks of BF16 over 32000 columns, 1.1 to 1.2 times.
// Experts, whose rows are an estimate: 1.02 for gate and up (208 tokens UINT4 286 -> 292 us without), and 1.08 where their blocks of 96 hold no fewer rows than those of 128 would
// (117 rows each, say): a Mixtral-8x7B layer of 130 to 1024 tokens 0.92 of the time in the geometric mean (0.79 .. 1.01); without the prices 468 tokens INT8 486 -> 548, UINT4 453 ->
// 513, with them 505 -> 477 and 458 -> 423.
constexpr float kPrice96[4] = {1.03f, 1.07f, 1.05f, 1.03f}; // INT8, BF16, NF4, UINT4

constexpr float kSplitStart[4] = {3.0f, 4.0f, 3.0f, 3.0f}, kSplitMb[4] = {0.3f, 0.35f, 0.3f, 0.3f}; // launch and megabytes of a split K's sum

// The same for activations staged through registers (K no whole number of 64, or more than 4 GB of them) and more than 256 rows: thresholds, as the
// constants above are those of other forms.  128-row tiles where they give every CU a block; below, K in parts while 64-row tiles give a CU
// less than two, and 32-row tiles where that is not enough.  With the model alone: INT8 450 x 4096 x 11040 71 -> 94 us, BF16 700 x 4096 x 4000 44
// -> 52.  BF16 weights, K a whole number of packed tiles: 2048 x 4096 x 11040 184 us, in the form for a ragged K 464, 1024 x 12288 x 4000
// 147 and 341.  false: up to 256 rows, where the model is the better one (1.03 to 2.7 times), and BF16 weights with a ragged K that do not fill the
// device with 128 x 256 (128 x 128 is 1.2 times slower than 64-row tiles there).
bool choose_staged_tile(SkinnyParams &p, int kind, int ktile, bool may_split) {
    const int cus = device_cu_count(), kt_n = (p.K + ktile - 1) / ktile;
    const long cols = (p.N + 127) / 128, large = (long)((p.N + 255) / 256) * ((p.M + 127) / 128), small = cols * ((p.M + 63) / 64);
    const bool bf16 = kind == XFTHIP_W_BF16;
    if (p.M <= 256) return false;
    if (large >= cus && (bf16 || p.M >= 512)) {
        p.tile = 4;
        return true;
    }
    if (bf16 && p.K % ktile != 0) return false;
    if (bf16 && p.M >= 512 && cols * ((p.M + 127) / 128) >= cus) {
        p.tile = 3;
        return true;
    }
    long want = 1;
    if (may_split && !p.gateup) {
        const long few = cols * ((p.M + 31) / 32);
        if (2 * few <= cus && kt_n >= 16) want = std::min({2L * cus / few, (long)kt_n / 8, 16L});
        else if (p.K >= 8192 && small < 2 * cus) want = std::min((2L * cus + small - 1) / small, (long)p.K / 2048);
        want = std::min(want, (long)(qgemm_split_bound() / ((size_t)p.M * p.N)));
    }
    if (want >= 2) {
        p.split_ktiles = (kt_n + (int)want - 1) / (int)want;
        p.ksplit = (kt_n + p.split_ktiles - 1) / p.split_ktiles;
    }
    p.tile = !bf16 && small * std::max(p.ksplit, 1) < 2 * cus ? 1 : 2;
    return true;
}

// own_sum: the caller adds the parts in a pass that it makes anyway
void choose_tile(SkinnyParams &p, int kind, int ktile, bool own_sum, bool may_split = true) {
    const int cus = device_cu_count(), kt_n = (p.K + ktile - 1) / ktile, cls = kind == XFTHIP_W_BF16 ? 1 : kind == XFTHIP_W_NF4 ? 2 : kind == XFTHIP_W_UINT4 ? 3 : 0;
    // activations straight into LDS: steps of 64 k, byte offsets of 32 bits
    const bool direct = p.K % 64 == 0 && (size_t)p.M * (size_t)p.lda * 2 < ((size_t)1 << 32);
    p.tile = 2, p.kgroups = 1, p.direct = 0;
    if (!direct && !p.rows_dev && choose_staged_tile(p, kind, ktile, may_split)) return;
    auto blocks_of = [&](const int rows) { // row blocks
        if (p.group) {
            // expected blocks of a weight whose rows scatter normally about their share: 1 + the chances that there are more than `rows`,
            // 2 `rows`, .. of them
            const float each = (float)p.M / (float)p.group_n, spread = sqrtf(each) + 0.1f * each;
            float blocks = 1.0f;
            for (int j = rows; (float)j < each + 4.0f * spread; j += rows) blocks += 0.5f * erfcf(((float)j - each) / (1.41421356f * spread));
            return (int)(blocks * (float)p.group_n + 0.999f);
        }
        return ((p.rows_dev && p.m_hint > 0 ? p.m_hint : p.M) + rows - 1) / rows;
    };
    float best = 1e30f;
    for (const TileCost &t : kTiles) {
        if (t.rows == 32 && kind == XFTHIP_W_BF16) continue; // (not built: two bytes a weight want more rows behind them)
        if (t.rows >= 96 && !direct) continue;
        if (t.kgroups == 2 && p.rows_dev) continue; // (not built)
        // (8 weights of 28672 x 4096 and 4096 x 14336 INT8 with 37 rows each: 386 us a layer in 32-row blocks, which read every weight tile twice,
        // 353 in 64-row ones)
        if (t.rows == 32 && p.group && p.M > 32 * p.group_n) continue;
        const int row_blocks = blocks_of(t.rows), col_blocks = (p.N + t.cols - 1) / t.cols;
        for (int want : {1, 2, 3, 4, 6, 8}) {
            if (want > 1 && (!may_split || p.gateup || p.K / want < 512)) break;
            int part = (kt_n + want - 1) / want; // packed tiles
            if (kind == XFTHIP_W_BF16) part = (part + 1) / 2 * 2; // (whole steps of 64)
            const int parts = (kt_n + part - 1) / part, span = parts > 1 ? part * ktile : p.K;
            if (parts > 1 && (size_t)parts * p.M * p.N > qgemm_split_bound()) break;
            const int band = band_rows(row_blocks, col_blocks * parts), bands = (row_blocks + band - 1) / band;
            const long blocks = ((long)bands * col_blocks * parts + 7) / 8 * 8 * band;
            float steps = (float)((span + 63) / 64);
            if (t.kgroups == 2) {
                // at most a block a CU, groups of whole packed tiles (in every part), deep enough to pay for their hand-over
                const int unit = 2 * (ktile > 64 ? ktile : 64);
                if (blocks > cus || p.K % unit || span % unit || steps < 48) continue;
                steps *= 0.5f;
            }
            // (with few blocks a 96-row tile's share of BF16 weights is too many bytes: 150 x 4096 x 11008 33 -> 45 us in 4 parts, 384 x 4096 x 22016 102 -> 118 whole)
            // (and 8 parts of K are dearer than the model has them: 384 x 14336 x 4096 INT8 57.6 us in 4, 64 in 8)
            if (t.rows == 96 && (parts > 4 || (kind == XFTHIP_W_BF16 && (parts > 1 || 2 * blocks < 3L * cus)))) continue;
            const long slots = (long)cus * t.resident, full = blocks / slots, rest = blocks - full * slots;
            float us = 7.0f + (float)full * (steps * (t.step[cls] + t.more[cls] * (float)(t.resident - 1)) + t.fixed);
            if (rest) {
                const float x = (float)rest / (float)cus, fullest = (float)((rest + cus - 1) / cus);
                us += steps * (x <= 1.0f ? t.step[cls] * (0.77f + 0.23f * x) : t.step[cls] + t.more[cls] * (0.55f * fullest + 0.45f * x - 1.0f)) + t.fixed;
            }
            if (parts > 1) us += (own_sum ? 0.0f : kSplitStart[cls]) + (own_sum ? 0.15f : kSplitMb[cls]) * 4e-6f * (float)parts * (float)p.M * (float)p.N;
            // (an expert's last block is half empty on average.  8 INT8 experts of width 2816 at width 2048, 700 tokens: 7 us more in 128 x 256 than in 64-row
            // blocks, which were to take 1 more; the layer 137 -> 129.  With down projections priced so as well, 256 tokens of the Mixtral shape
            // lose 0.7 %)
            if (p.group && p.gateup && t.rows == 128) us *= 1.05f;
            if (t.rows == 96) us *= !p.group ? kPrice96[cls] : 96 * row_blocks >= 128 * blocks_of(128) ? 1.08f : p.gateup ? 1.02f : 1.0f;
            if (us < best) {
                best = us;
                p.tile = t.rows == 32 ? 1 : t.rows == 64 ? 2 : t.rows == 96 ? 5 : t.cols == 128 ? 3 : 4;
                p.kgroups = t.kgroups, p.direct = t.rows >= 96;
                p.ksplit = parts > 1 ? parts : 0, p.split_ktiles = part;
            }
        }
    }
}

} // namespace

// Partial results of the K split: one buffer per stream and device (stream_scratch), allocated once at its upper
// bound (64 KB of results a CU in 4 parts: 67 MB on 256 CUs; a split that needs more is not taken), so
// nothing is allocated or freed on a stream once its buffer exists.  Launches on one stream are ordered; launches
// on different streams work in different buffers.
size_t qgemm_split_bound() { return (size_t)device_cu_count() * 65536; }

bool qgemm_split_usable(hipStream_t stream) {
    // (the null stream cannot be captured, and must not be asked: while another one is, the answer is an error, which the launch's own check would report)
    if (stream == nullptr) return true;
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(stream, &status) != hipSuccess) {
        (void)hipGetLastError();
        return true;
    }
    if (status == hipStreamCaptureStatusNone) return true;
    return stream_scratch_held(kScratchGemmSplit, stream, qgemm_split_bound() * sizeof(float));
}

int qgemm_split_reserve(hipStream_t stream, float **out) {
    void *p = nullptr;
    if (int rc = stream_scratch(kScratchGemmSplit, stream, qgemm_split_bound() * sizeof(float), false, &p)) return rc;
    if (out) *out = (float *)p;
    return 0;
}

void qgemm_mfma_form(int kind, SkinnyParams &p) {
    choose_tile(p, kind, ktile_of(kind), false);
}

int qgemm_mfma(const PackedWeight &pw, const SkinnyParams &p0, hipStream_t stream, int *parts, const float **part) {
    SkinnyParams p = p0;
    p.packed = pw.packed;
    p.scale = pw.scale;
    p.zero = pw.zero;
    p.KT = pw.KT;
    p.NTILES = pw.NTILES;
    p.K = pw.K;
    p.N = pw.N;
    p.ksplit = 0, p.split_ktiles = 0, p.split_part = nullptr;
    const int ktile = ktile_of(pw.kind), kt_n = (pw.K + ktile - 1) / ktile;
    choose_tile(p, pw.kind, ktile, parts != nullptr);
    if (p.ksplit > 1 && !qgemm_split_usable(stream)) p.ksplit = 0, choose_tile(p, pw.kind, ktile, false, false);
    if (p.ksplit > 1) {
        if ((size_t)p.ksplit * p.M * p.N > qgemm_split_bound()) p.ksplit = 0; // cannot happen within the bound; stay correct anyway
        else if (int rc = qgemm_split_reserve(stream, &p.split_part)) return rc;
    }
    if (p.ksplit <= 1) p.ksplit = 0;
    int (*kernel)(const SkinnyParams &, hipStream_t) = nullptr;
    switch (pw.kind) {
        case XFTHIP_W_INT8: kernel = p.zero ? qgemm_mfma_int8z : qgemm_mfma_int8; break;
        case XFTHIP_W_UINT4: kernel = qgemm_mfma_uint4; break;
        case XFTHIP_W_NF4: kernel = qgemm_mfma_nf4; break;
        case XFTHIP_W_BF16: kernel = qgemm_mfma_bf16; break;
        default: set_error("qgemm_mfma: weight kind %d not supported", pw.kind); return 2;
    }
    XFT_REQUIRE(kernel, "qgemm_mfma: this library was built for BF16 weights only");
    const int rc = kernel(p, stream);
    if (rc || p.ksplit <= 1) return rc;
    if (parts) {
        *parts = p.ksplit, *part = p.split_part;
        return 0;
    }
    const size_t outs = (size_t)p.M * p.N;
    if (p.N % 4 == 0) // the parts are [M][N] fp32 in a 256-byte aligned buffer: 16-byte loads need only N % 4 == 0
        hipLaunchKernelGGL(qgemm_split_finish_kernel<4>, dim3((unsigned)((outs / 4 + 255) / 256)), dim3(256), 0, stream, p);
    else
        hipLaunchKernelGGL(qgemm_split_finish_kernel<1>, dim3((unsigned)((outs + 255) / 256)), dim3(256), 0, stream, p);
    XFT_CHECK_HIP(hipGetLastError());
    return 0;
}

} // namespace xfthip
