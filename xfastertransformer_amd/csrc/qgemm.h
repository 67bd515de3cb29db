// Parameter block shared by the weight-only GEMM kernels and their C-ABI entry points.
#pragma once
#include "common.h"
#include "kvcache.h"

namespace xfthip {

struct GroupWeight { // one weight of a grouped launch, in device memory
    const uint8_t *packed;
    const float *scale;
    const float *zero;
};

// Device memory as such: pointers read from memory are generic ones to the compiler, and a load through them waits, and is waited for, like an access to LDS
// as well, so that every operand read from there held up the weights on their way (experts, whose weights come from a table: INT8, 256 tokens of the Mixtral shape
// 400 -> 381 us, 1000 895 -> 843, UINT4, 100 tokens 203 -> 189).
#define XFT_GLOBAL __attribute__((address_space(1)))
inline __device__ const XFT_GLOBAL uint8_t *global_bytes(const uint8_t *p) { return (const XFT_GLOBAL uint8_t *)(uintptr_t)p; }

struct SkinnyParams {
    const uint8_t *packed;
    const float *scale;
    const float *zero;
    int KT, NTILES, K, N, M;
    const uint16_t *A; // bf16
    int lda;
    void *C;
    int ldc, c_dtype;
    int epi;
    const float *bias; // [N]; gateup: of the gate columns, behind them of the others
    const void *res;
    int ldres, res_dtype;
    float gamma;
    int gateup; // 1: combine tile pairs as silu(gate)*up, N counts cat columns; 2: as clamped_glu (below)
    float glu_limit, glu_alpha; // gateup == 2
    int nblocks; // column blocks of the launch (set by the launcher)
    // K split of the M > 32 kernel (few rows against few columns and a deep K): workgroup row blockIdx.y
    // multiplies k tiles [y * split_ktiles, (y + 1) * split_ktiles) and writes its scaled partial result as
    // fp32 [M][N] into split_part + y * M * N; a second kernel adds the parts in order and applies the epilogue
    int ksplit, split_ktiles;
    float *split_part;
    // M > 32 kernel, host-side row count: the block tile (1: 32 rows x 128 columns, 2: 64 x 128, 3: 128 x 128, 4: 128 x 256, 5: 96 x 256), its K groups
    // a workgroup, whether the activations go straight into LDS (tiles 3, 4 and 5); chosen by qgemm_mfma.  band: row blocks a band of the launch
    int tile, kgroups, direct, band;
    // Row count known on the device only (the experts of a sparse MLP): when rows_dev is set the kernels read
    // {rows, first row of A, first row of C} from it, M is only the upper bound that sizes the grid, and m_hint
    // (0 = M) is the row count the host expects, used where it chooses between forms.  No residual epilogues.
    const int *rows_dev;
    int m_hint;
    // Several weights of one shape and kind behind one launch: weight e multiplies the rows
    // that record e of rows_dev (records rows_stride ints apart) names; M bounds the sum of their rows, and their
    // rows of C must tile [0, sum of rows) without gaps.
    const GroupWeight *group;
    int group_n, rows_stride;
    const int *a_rows; // groups only, or null: row r of A (record offset included) is row a_rows[r] of it

    // ---- fusions of the decode step (M <= 4, skinny kernel only) ----
    // RMSNorm prologue: when norm_x is set, A is ignored and every workgroup normalises the M rows
    // of norm_x (fp32, row pitch ldx) with norm_w / norm_eps into LDS itself (same arithmetic as
    // the rmsnorm kernel, bf16 result) while its first weight tiles are in flight.
    const float *norm_x;
    int ldx;
    const float *norm_w;
    float norm_eps;
    // RoPE + cache append epilogue of the QKV projection (one new token per sequence, FP16 cache):
    // column tiles are paired (d, d + 64) within a head, the rotated query goes to C as bf16
    // (row pitch ldc, q_heads * 128 columns), rotated keys and the values go to the cache at
    // position pos_dev[m] (or pos_host when pos_dev is null).  The tables hold 64 entries a row.
    int rope;
    const float *cosT, *sinT;
    const int *pos_dev;
    int pos_host;
    int qH, kvH;
    KvView kv;
};

// The clamped gated unit: g = min(gate, limit), u = clamp(up, -limit, limit), g * sigmoid(alpha g) * (u + 1)
__device__ inline float clamped_glu(float gate, float up, float limit, float alpha) {
    const float g = fminf(gate, limit), u = fminf(fmaxf(up, -limit), limit);
    return g / (1.0f + fast_exp(-alpha * g)) * (u + 1.0f);
}

// Row blocks are walked in bands of at most 8 (qgemm_mfma_impl.h), `units` units of work a band.  The bands are of one height, the
// one that leaves the XCD with the most units the least to do (3072 columns in 256s, 19 row blocks: three bands of 7 are 36 units,
// five for some XCDs, 35 blocks on 32 CUs; four of 5 are 48, six each, 30 blocks), and no band of a few rows is padded to 8 with
// workgroups that leave at once.  Those do harm: an XCD hands its workgroups to its four shader engines in turn, whatever they
// do there, so that 5 working ones of 8 put two on the first engine and one on each other (600 x 12288 x 4096 INT8, 240 blocks of
// two K groups on 256 CUs: over 100 us against 65).
__host__ __device__ inline int band_rows(int nblocks_m, int units) {
    const int bands = (nblocks_m + 7) / 8;
    int best = nblocks_m > 0 ? (nblocks_m + bands - 1) / bands : 1, least = (bands * units + 7) / 8 * best;
    for (int n = bands + 1; n <= bands + 3; ++n) {
        const int rows = (nblocks_m + n - 1) / n, load = (n * units + 7) / 8 * rows;
        if (load < least) best = rows, least = load;
    }
    return best;
}

// The form of a product of up to 32 rows without prologue and RoPE, K of whole tiles: column tiles a block, k tiles a load batch, K slices (waves)
struct SkinnyForm {
    int nt, u, kslices;
};
// k tiles a load batch of a block of nt column tiles and mt 16-row tiles: what the kernels are built with and what skinny_form counts slices in
// (but BF16 single tiles that are a CU's only block: skinny_form)
constexpr int skinny_batch(int kind, int mt, bool group, int nt) {
    if (kind == XFTHIP_W_UINT4 || kind == XFTHIP_W_NF4 || nt > 3) return 1;
    const bool int8 = kind == XFTHIP_W_INT8;
    if (nt == 3) return mt == 1 ? 1 : 2;
    if (mt == 1) return nt == 1 ? (int8 || group ? 4 : 2) : (group && !int8 ? 4 : 2);
    return nt == 2 && int8 && group ? 1 : 2;
}
// Products of 4-bit codes whose activation rows go straight into LDS (mt 16-row tiles): all that are staged, but UINT4 at up to 16 rows, where it gains 2 % in the mean and
// loses up to 8 % (skinny_form has the figures)
constexpr bool skinny_dma(int kind, int mt) { return kind == XFTHIP_W_NF4 || (kind == XFTHIP_W_UINT4 && mt == 2); }
// rows that lie 4 GB apart, out of reach of that form's 32-bit offsets in bytes: the form for a ragged K takes them, which counts in elements (gemm_rows: 8 GB)
inline bool skinny_far(int kind, const SkinnyParams &p) {
    return p.M > 4 && !p.group && skinny_dma(kind, p.M > 16 ? 2 : 1) && (size_t)p.M * (size_t)p.lda * 2 >= (size_t)1 << 32;
}
SkinnyForm skinny_form(int kind, const SkinnyParams &p);
int qgemm_skinny(const PackedWeight &pw, const SkinnyParams &p, hipStream_t stream); // M <= 32
bool skinny_can_fuse_norm(const PackedWeight &pw, int M); // may SkinnyParams::norm_x be used
// any M, built for M > 32; parts / part: as in gemm_grouped_rows_dev
int qgemm_mfma(const PackedWeight &pw, const SkinnyParams &p, hipStream_t stream, int *parts = nullptr, const float **part = nullptr);
void qgemm_mfma_form(int kind, SkinnyParams &p); // the tile, K groups and K parts it takes, into p (ksplit: 0 where K is whole)
// the K-split workspace of qgemm_mfma launches on `stream` (allocated on the stream's first call: before a capture, say)
int qgemm_split_reserve(hipStream_t stream, float **out = nullptr);
size_t qgemm_split_bound(); // its floats
// may a launch on `stream` use it: not while the stream is captured without having it (allocating would end the capture)
bool qgemm_split_usable(hipStream_t stream);
// xfthip_gemm / xfthip_gemm_gateup_silu (by the weight's flag) with the row count in device memory: rows_dev =
// {rows, first row of A, first row of C}, at most m_max rows, about m_hint expected; plain epilogue only
int gemm_rows_dev(xfthip_weight_t w, int m_max, int m_hint, const int *rows_dev, const void *A, int lda, void *C, int ldc, int c_dtype,
        hipStream_t stream);

// The same for n_group weights of one shape behind one launch: table_dev holds their device pointers, record e
// of rows_dev (rows_stride ints apart) the rows of weight e; rows_max bounds the sum of the rows, rows_each_max the
// rows of one weight (up to 32 of those: the few-row kernel, one grid row a weight; more: the tiled kernel, row
// blocks numbered across the weights); the weights' rows of C tile [0, sum of rows).  a_rows: as in SkinnyParams.
// glu_alpha > 0: gate / up weights combine as clamped_glu instead of as SwiGLU.  parts / part (fp32 results only): where K was split, the parts
// stay as they are, *parts of [rows_max][N] one after the other from *part on, until the stream's next product; else C is written, *parts = 1.
int gemm_grouped_rows_dev(const xfthip_weight_t *w, int n_group, const GroupWeight *table_dev, int rows_max, int rows_each_max,
        const int *rows_dev, int rows_stride, const void *A, int lda, void *C, int ldc, int c_dtype, hipStream_t stream,
        const int *a_rows = nullptr, float glu_limit = 0.0f, float glu_alpha = 0.0f, int *parts = nullptr, const float **part = nullptr);

int gemm_w8a8_from_bf16(xfthip_weight_t w, int M, const void *A, int lda, void *C, int ldc, int c_dtype, int epilogue,
        const float *bias, const void *res, int ldres, int res_dtype, float gamma, hipStream_t stream);

} // namespace xfthip
