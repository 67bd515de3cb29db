// Dequant-fused weight-only GEMM for few activation rows (M <= 32): the decode-time shape.
// Replaces MMHelper::compute* (reference src/utils/matmul_helper.h:565-1705) for
// INT8 / UINT4 / NF4 / BF16 weights against bf16 activations.  The kernel lives in
// qgemm_skinny_impl.h; this file checks the fused options, picks the weight kind and the form.
#include "qgemm.h"

namespace xfthip {

// weak: a library for models with BF16 weights only is built without the quantised kinds (build.py)
__attribute__((weak)) int qgemm_skinny_int8(const SkinnyParams &p, hipStream_t stream);
__attribute__((weak)) int qgemm_skinny_uint4(const SkinnyParams &p, hipStream_t stream);
__attribute__((weak)) int qgemm_skinny_nf4(const SkinnyParams &p, hipStream_t stream);
int qgemm_skinny_bf16(const SkinnyParams &p, hipStream_t stream);

// LDS of the RMSNorm prologue: M rows of K + 8 bf16 values
static inline size_t skinny_norm_lds_bytes(int M, int K) {
    return (size_t)M * (K + 8) * 2;
}

bool skinny_can_fuse_norm(const PackedWeight &pw, int M) {
    return M <= 4 && pw.kind != XFTHIP_W_W8A8 && pw.KT * ktile_of(pw.kind) == pw.K && pw.K % 4 == 0
            && skinny_norm_lds_bytes(M, pw.K) <= (size_t)36 * 1024;
}

// What sets the time is the CU with the most column tiles: blocks are spread over the CUs in turn, so that it is w = ceil(blocks / CUs) blocks of nt
// tiles.  A tile costs least in blocks of two (an activation fragment serves both; wider blocks lose some of that to registers), a block half a
// tile more for its sums over the waves.  All blocks of a CU run side by side: 8 waves between them keep enough loads in flight (more K
// slices only add sums), two a block at least.  BF16 at up to 16 rows: single tiles, whose stream alone is 32 KB a block.
// Timed over 20 shapes of 512 .. 32000 columns x 1408 .. 14336 deep, six row counts, four kinds, all forms: 0.96 .. 0.99 of the best form on
// average.  Against two tiles (3 .. 6 at 17 .. 32 rows) in 8 slices throughout, geometric mean at up to 4 / 16 / 32 rows: UINT4 1.13 / 1.16 /
// 1.07 times as fast, NF4 1.12 / 1.14 / 1.08, INT8 1.04 / 1.08 / 1.07, BF16 1.03 / 1.03 / 1.05; UINT4 24 x 4096 x 28672 30 -> 22 us, 6 rows
// 25 -> 15.6, 16 x 8192 x 10240 19 -> 14.
// More than 8 tiles a CU, where the blocks come in rounds anyway: the form that was best over 55296 .. 151936 columns (UINT4 16 x 4096 x 128256
// 101 -> 52 us, INT8 32 rows 126 -> 101, NF4 6 rows 115 -> 74, BF16 6 rows 166 -> 152).
// Several weights behind one launch: the same over the columns of those that have rows, as many as there are rows at most.  8 weights each of
// 28672 x 4096 and 4096 x 14336, a layer of 10 / 32 tokens: UINT4 224 / 306 -> 142 / 207 us, NF4 284 / 384 -> 200 / 280,
// INT8 255 / 333 -> 214 / 276, BF16 400 / 501 -> 394 / 484.
SkinnyForm skinny_form(int kind, const SkinnyParams &p) {
    const bool four = kind == XFTHIP_W_UINT4 || kind == XFTHIP_W_NF4;
    const int cus = device_cu_count(), mt = p.M <= 16 ? 1 : 2;
    const int weights = !p.group ? 1 : p.m_hint < 1 ? 1 : p.m_hint < p.group_n ? p.m_hint : p.group_n;
    auto form = [&](int nt, int kslices) { // a batch a slice at least
        const int u = skinny_batch(kind, mt, p.group != nullptr, nt), batches = p.KT / u;
        kslices = kslices < 8 ? kslices : 8;
        kslices = kslices < batches ? kslices : batches;
        return SkinnyForm {nt, u, kslices > 1 ? kslices : 1};
    };
    auto per_cu = [&](int nt) { return ((p.NTILES + nt - 1) / nt * weights + cus - 1) / cus; };
    const long tiles = (long)p.NTILES * weights;
    if (p.M > 4 && !p.group && skinny_dma(kind, mt)) {
        // Rows straight into LDS, 16 KB a wave (8 at up to 16 rows): eight waves a CU have room, and it needs them all, so that a CU's blocks share them; wide blocks hold no
        // rows in registers.  Against rows staged through registers (with v_and_or_b32 in both), 101 shapes of 1024 .. 151936 columns x 256 .. 28672 deep: UINT4 24 and 32 rows 0.92 of the time
        // in the geometric mean (0.77 .. 1.02; 24 x 4096 x 28672 with SwiGLU 21.4 -> 18.7 us), NF4 0.90 (0.75 .. 1.02), at up to 16 rows 0.92 (0.78 .. 1.03); within 0.5 to 1.3 % of the
        // best of 20 forms in the mean.  With half the waves in blocks of six tiles, and 0.8 of a tile a block, which this rule had first, up to 1.23: NF4 24 x 3584 x
        // 37888 with SwiGLU 33.5 -> 40.4, now 28.5, UINT4 32 x 7168 x 52192 58.5 -> 68.9, now 56.0.
        // NF4 at up to 16 rows, more than 12 tiles a CU: 16 x 4096 x 128256 77 us in three tiles, 73 staged, 68.7 in four.
        if (mt == 1 && tiles > 12L * cus) return SkinnyForm {4, 1, p.KT > 1 ? 2 : 1};
        int best = p.gateup ? 2 : 1;
        float least = 1e30f;
        for (int n : {1, 2, 3, 4, 6}) {
            if (p.gateup && n % 2) continue;
            const float tile = mt == 2 || n < 4 ? 1.0f : n == 4 ? 1.1f : 1.2f;
            const float cost = (float)per_cu(n) * ((float)n * tile + (mt == 2 ? 1.2f : 0.4f));
            if (cost < least) least = cost, best = n;
        }
        const int w = per_cu(best), slices = w == 1 ? 8 : w == 2 ? 4 : 2;
        return SkinnyForm {best, 1, slices < p.KT ? slices : p.KT};
    }
    // (two slices against eight: 3 % faster at K = 4096, 2 % slower at 2048)
    if (kind == XFTHIP_W_BF16 && p.group && mt == 1) return form(p.gateup ? 2 : 1, p.gateup && p.K >= 4096 ? 2 : 8);
    if (p.group && tiles >= 8 * cus) { // K slices by the depth
        if (four && mt == 1) return form(p.M <= 4 ? 2 : 4, p.KT < 32 ? 4 : p.KT / 8);
        if (four) return form(4, p.KT / 16);
        if (kind == XFTHIP_W_INT8) return mt == 1 ? form(2, p.KT / 8) : form(2, 4);
        return form(2, 2);
    }
    if (tiles > 8 * cus) {
        // (a shallow K goes by its own counts, for no reason that is known: in the forms for a deeper one INT8 8 rows of 1024 x 65024 17.6 us, of
        // 2048 x 151936 55.0, here 15.3 and 49.9; BF16 32 rows of 1024 x 65024 35.6 and 29.4.  INT8 8 rows of 8192 x 55296: 83 us in 8 slices, 74 in one;
        // 32 rows of 3584 x 100000 79 in 3, 77 in 4, of 8192 x 55296 92 and 102)
        const bool shallow = p.K <= 2048;
        if (mt == 2 && kind == XFTHIP_W_BF16 && shallow) return form(2, p.K < 2048 ? 2 : 1);
        if (mt == 2) return form(4, four ? 2 : kind == XFTHIP_W_INT8 ? (p.KT > 32 && p.KT % 32 ? 4 : 3) : 1);
        if (four) return form(4, 4);
        if (shallow && (kind == XFTHIP_W_INT8 || p.M > 8 || p.K > 1024)) return form(2, 3);
        // (BF16, 16 rows of 128256 columns: single tiles in 8 slices 199 us, 171 before, 166 in this form)
        if (kind == XFTHIP_W_BF16 && p.M > 8) return form(2, 1);
        return form(kind == XFTHIP_W_INT8 || p.gateup ? 2 : 1, kind == XFTHIP_W_INT8 && p.K >= 8192 ? 1 : 8);
    }
    int nt = p.gateup ? 2 : 1;
    if (kind != XFTHIP_W_BF16 || mt == 2) {
        float least = 1e30f;
        for (int n : {1, 2, 3, 4, 6}) {
            if ((p.gateup && n % 2) || (n >= 4 && mt == 1) || (n % 3 == 0 && p.group)) continue;
            const int w = per_cu(n);
            // (17 .. 32 rows, two blocks of four tiles on a CU: well for 4-bit codes and a deep INT8 K (32 rows x 27648 x 5120 41.6 -> 36.1 us), 1.2
            // times the time of four blocks of two for the others)
            const bool dear = n == 4 && w > 1 && !four && !(kind == XFTHIP_W_INT8 && p.KT >= 80);
            const float tile = n == 1 ? 1.2f : n == 2 ? 1.0f : dear ? 1.3f : 1.1f;
            const float cost = (float)w * ((float)n * tile + 0.5f);
            if (cost < least) least = cost, nt = n;
        }
    }
    // A BF16 tile alone on its CU, 13 .. 16 rows: batches of four k tiles in four slices, the bytes in flight of batches of two in eight with half the waits (and two
    // sums a wave, so that an fp32 sum is as short).  16 rows, K x N: 5632 x 2048 10.2 -> 9.7 us, 11008 x 4096 20.8 -> 19.6, 8192 x 3072 14.3 -> 13.8, 14336 x 4096 26.2
    // -> 24.9, 23.5 -> 22.0 where the weights lie in the Infinity Cache.  With fewer rows only where most CUs have a tile and a slice is a whole number of two
    // batches, or many of them: 8 rows of 4096 x 4096 8.4 -> 8.1, 11008 x 4096 20.5 -> 19.9, 8192 x 3072 13.1 -> 12.3, but 4480 x 4096 8.9 -> 9.1, 4096 x 512 5.7 -> 5.9,
    // 5 of 32768 x 64 25.4 -> 26.5 (8 of 14336 x 4096 22.5 in both, 19.4 -> 19.9 out of the Infinity Cache).  Not for a K of half a batch, a shallow one, up to 4 rows or two tiles a CU, which lose: 16 rows of 4128 x 4096 9.4 -> 9.6, of 2048 x
    // 2048 4.6 -> 4.8, 3 of 14336 x 4096 18.7 -> 19.4; 1 of 4096 x 6144 10.5 -> 11.0.
    if (kind == XFTHIP_W_BF16 && mt == 1 && nt == 1 && !p.group && p.K >= 4096 && p.KT % 4 == 0 && per_cu(1) == 1) {
        const bool filled = 4 * p.NTILES >= 3 * cus && (p.KT % 32 == 0 || p.K >= 8192);
        if (p.M > (filled ? 6 : 12)) return SkinnyForm {1, 4, 4};
    }
    // (BF16, four blocks of two tiles on a CU: one slice each, 32 rows x 28672 x 8192 101 -> 88 us, with SwiGLU 8 rows x 28672 x 4096 1.07 times as fast)
    const int least = kind == XFTHIP_W_BF16 ? 1 : 2, slices = kind == XFTHIP_W_BF16 && nt == 2 && per_cu(nt) > 2 ? 1 : 8 / per_cu(nt);
    return form(nt, slices > least ? slices : least);
}

int qgemm_skinny(const PackedWeight &pw, const SkinnyParams &p0, hipStream_t stream) {
    SkinnyParams p = p0;
    if (p.group && (p.norm_x || p.rope || !p.rows_dev || (pw.KT * ktile_of(pw.kind) != pw.K && pw.kind != XFTHIP_W_BF16))) {
        set_error("qgemm_skinny: a group of weights needs device row records and K a whole number of weight tiles (BF16 weights: any K), and "
                  "takes no norm prologue or RoPE epilogue");
        return 2;
    }
    if (p.norm_x && !skinny_can_fuse_norm(pw, p.M)) {
        set_error("qgemm_skinny: RMSNorm prologue not available for M=%d K=%d kind=%d", p.M, pw.K, pw.kind);
        return 2;
    }
    if (p.rope && (p.M > 32 || p.M > p.kv.B || p.kvH != p.kv.H || p.gateup || (p.qH + 2 * p.kvH) * 128 != pw.N || p.kv.int8 != 0 || p.kv.D != 128
                || (p.M > 16 && p.norm_x))) {
        set_error("qgemm_skinny: RoPE / cache-append epilogue needs M <= 32 rows (one per cache row), head size 128, an FP16 cache and a "
                  "[K, (q+2kv)*128] weight");
        return 2;
    }
    p.packed = pw.packed;
    p.scale = pw.scale;
    p.zero = pw.zero;
    p.KT = pw.KT;
    p.NTILES = pw.NTILES;
    p.K = pw.K;
    p.N = pw.N;
    int (*quantised)(const SkinnyParams &, hipStream_t) = nullptr;
    switch (pw.kind) {
        case XFTHIP_W_INT8: quantised = qgemm_skinny_int8; break;
        case XFTHIP_W_UINT4: quantised = qgemm_skinny_uint4; break;
        case XFTHIP_W_NF4: quantised = qgemm_skinny_nf4; break;
        case XFTHIP_W_BF16: return qgemm_skinny_bf16(p, stream);
        default: set_error("qgemm_skinny: weight kind %d not supported", pw.kind); return 2;
    }
    XFT_REQUIRE(quantised, "qgemm_skinny: this library was built for BF16 weights only");
    return quantised(p, stream);
}

} // namespace xfthip
