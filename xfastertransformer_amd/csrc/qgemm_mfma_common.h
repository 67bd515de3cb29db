// What the kernels of the weight-only GEMM for many activation rows share (qgemm_direct_impl.h, qgemm_mfma_impl.h): which block a workgroup computes and how
// its results leave.
#pragma once
#include <type_traits>

#include "qgemm.h"

namespace xfthip {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

union MFrag {
    bf16x8 v;
    uint32_t u[4];
    u32x4 q;
};

__device__ inline uint32_t pack_hi16_m(float lo, float hi) {
    return __builtin_amdgcn_perm(f2u(hi), f2u(lo), 0x07060302u);
}

__constant__ float c_nf4_big[16] = XFTHIP_NF4_CODE_VALUES;

__device__ inline float silu_big(float x) {
    return x / (1.0f + fast_exp(-x));
}

// The block of workgroup blockIdx.x: column block nb, first row m0 and, in p, the operands and results of its K part and of its weight; false: none.
template <int ROWS, int PACKED_K, bool DEVROWS>
__device__ __forceinline__ bool take_block(SkinnyParams &p, const int nblocks_n, int nblocks_m, const int lane, int &nb, int &m0) {
    const int part_rows = p.M; // rows of a K part: the host's bound, also when the device knows fewer
    // workgroup -> (K part, column block, row block).  Row blocks are walked in bands (band_rows); a unit of work is one
    // (band, K part, column block): its workgroups share the column block's weights.  Workgroup ids go round the 8
    // XCDs in launch order, so the units are dealt out to the XCDs one by one - an XCD runs the workgroups of a unit
    // next to each other (the weights pass through its L2 once) and its units follow each other column block by column
    // block inside a band (the band's activation rows stay in its L2 while the weights stream past them) - and the
    // XCDs carry the same load whatever the number of column blocks (43 blocks of 256 columns dealt out block by block
    // would give three XCDs 6 and five XCDs 5).
    // Row counts on the device: the row blocks that are there are numbered, so that all workgroups past them come last.
    int group_upto = 0; // (lane e of every wave, groups) row blocks of the weights up to and including weight e of its 64
    if constexpr (DEVROWS) {
        if (p.group) {
            nblocks_m = 0;
            for (int e0 = 0; e0 < p.group_n; e0 += 64) {
                int n = e0 + lane < p.group_n ? (p.rows_dev[(e0 + lane) * p.rows_stride] + ROWS - 1) / ROWS : 0;
#pragma unroll
                for (int off = 1; off < 64; off <<= 1) {
                    const int up = __shfl_up(n, off, 64);
                    n += lane >= off ? up : 0;
                }
                group_upto = n; // (of the last 64)
                nblocks_m += __builtin_amdgcn_readlane(n, 63);
            }
        } else if (p.rows_dev) {
            p.M = p.rows_dev[0] < part_rows ? p.rows_dev[0] : part_rows;
            nblocks_m = (p.M + ROWS - 1) / ROWS;
        }
    }
    int mb, part;
    {
        const int parts = p.ksplit > 1 ? p.ksplit : 1;
        const int BAND = DEVROWS ? band_rows(nblocks_m, parts * nblocks_n) : p.band; // (its divisions: not in every workgroup where the host can)
        const int id = blockIdx.x, xcd = id & 7, slot = id >> 3; // gridDim.x is a multiple of 8
        const int nbands = (nblocks_m + BAND - 1) / BAND;
        const int units = nbands * parts * nblocks_n;
        const int unit = (slot / BAND) * 8 + xcd;
        if (unit >= units) return false;
        const int band = unit / (parts * nblocks_n), rem = unit - band * (parts * nblocks_n);
        part = rem / nblocks_n;
        nb = rem - part * nblocks_n;
        mb = band * BAND + slot % BAND;
        if (mb >= nblocks_m) return false;
    }
    int c_row = 0, part_row = 0; // first row of this GEMM in C and in a K part
    if constexpr (DEVROWS) {
    if (p.group) {
        // several weights of one shape behind one launch: the row blocks of all of them are numbered in a
        // row, weight after weight, by their device-side row counts
        int e = 0, first = 0;
        if (p.group_n <= 64) {
            const unsigned long long before = __builtin_amdgcn_ballot_w64(group_upto <= mb);
            e = __builtin_popcountll(before); // (group_upto is ascending over the lanes)
            first = e ? __builtin_amdgcn_readlane(group_upto, e - 1) : 0;
        } else {
            for (; e < p.group_n; ++e) {
                const int nblk = (p.rows_dev[e * p.rows_stride] + ROWS - 1) / ROWS;
                if (mb < first + nblk) break;
                first += nblk;
            }
        }
        if (e >= p.group_n) return false;
        mb -= first;
        const int *rec = p.rows_dev + e * p.rows_stride;
        p.M = rec[0];
        if (p.a_rows) p.a_rows += rec[1];
        else p.A += (size_t)rec[1] * p.lda;
        c_row = part_row = rec[2];
        p.packed = p.group[e].packed;
        p.scale = p.group[e].scale;
        p.zero = p.group[e].zero;
    } else if (p.rows_dev) {
        p.A += (size_t)p.rows_dev[1] * p.lda;
        c_row = p.rows_dev[2]; // the K parts hold local rows, the kernel that adds them shifts
    }
    p.C = (char *)p.C + (size_t)c_row * p.ldc * (p.c_dtype == XFTHIP_F32 ? 4 : 2);
    }
    if (p.ksplit > 1) {
        // this workgroup owns a range of k tiles: shift the operands to it, the result goes to its part
        const int kt0 = part * p.split_ktiles;
        const int k_left = p.K - kt0 * PACKED_K, k_span = p.split_ktiles * PACKED_K; // (split_ktiles counts packed tiles)
        p.packed += (size_t)kt0 * 1024;
        p.A += (size_t)kt0 * PACKED_K;
        p.K = k_left < k_span ? k_left : k_span;
        p.C = p.split_part + ((size_t)part * part_rows + part_row) * p.N;
        p.ldc = p.N;
        p.c_dtype = XFTHIP_F32;
        p.epi = XFTHIP_EPI_NONE;
    }
    m0 = mb * ROWS;
    return !DEVROWS || m0 < p.M; // (fewer rows than the grid was sized for: the whole workgroup leaves)
}

// A wave's results on their way out: rows of fp32 in an LDS patch of its own
struct FlushRows {
    const unsigned char *patch;
    int pitch, lane;
    bool c_wide, res_wide; // 16-byte accesses to C / the residual
};
__device__ inline FlushRows flush_target(const SkinnyParams &p, const unsigned char *patch, int pitch, int lane) {
    FlushRows to = {patch, pitch, lane, false, false};
    to.c_wide = (((size_t)p.C | ((size_t)p.ldc * (p.c_dtype == XFTHIP_F32 ? 4 : 2))) & 15) == 0;
    to.res_wide = (((size_t)p.res | ((size_t)p.ldres * (p.res_dtype == XFTHIP_F32 ? 4 : 2))) & 15) == 0;
    return to;
}
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}
// the 32 rows of the patch, strip_cols wide, are rows row0 .. of the result and go to output columns col0 .. col_end - 1
template <int EPI>
__device__ __forceinline__ void flush_rows(const FlushRows &to, const SkinnyParams &p, int row0, int col0, int strip_cols, int col_end) {
    constexpr bool HAS_RES = EPI == XFTHIP_EPI_RESMUL || EPI == XFTHIP_EPI_RESIDENTIAL || EPI == XFTHIP_EPI_RESEXT;
    wave_sync();
    const int cpr = strip_cols >> 3; // 8-column chunks a row: 2, 4 or 8
    const int cpr_log2 = __builtin_ctz(cpr);
    for (int idx = to.lane; idx < 32 * cpr; idx += 64) {
        const int r = idx >> cpr_log2, ch = idx & (cpr - 1);
        const int row = row0 + r;
        const int c = col0 + 8 * ch;
        if (row >= p.M || c >= col_end) continue;
        const float *src = (const float *)(to.patch + r * to.pitch) + 8 * ch;
        const f32x4 lo = *(const f32x4 *)src, hi = *(const f32x4 *)(src + 4);
        float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        const bool full = c + 8 <= col_end;
        if constexpr (HAS_RES) {
            const size_t ri = (size_t)row * p.ldres + c;
            float rv[8];
            if (full && to.res_wide) {
                if (p.res_dtype == XFTHIP_F32) {
                    const f32x4 r0 = *(const f32x4 *)((const float *)p.res + ri), r1 = *(const f32x4 *)((const float *)p.res + ri + 4);
                    rv[0] = r0[0], rv[1] = r0[1], rv[2] = r0[2], rv[3] = r0[3], rv[4] = r1[0], rv[5] = r1[1], rv[6] = r1[2], rv[7] = r1[3];
                } else {
                    const u32x4 rr = *(const u32x4 *)((const uint16_t *)p.res + ri);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint16_t b0 = (uint16_t)rr[e], b1 = (uint16_t)(rr[e] >> 16);
                        rv[2 * e] = p.res_dtype == XFTHIP_BF16 ? bf16_to_f32(b0) : fp16_bits_to_f32(b0);
                        rv[2 * e + 1] = p.res_dtype == XFTHIP_BF16 ? bf16_to_f32(b1) : fp16_bits_to_f32(b1);
                    }
                }
            } else {
#pragma unroll
                for (int e = 0; e < 8; ++e) rv[e] = c + e < col_end ? load_as_f32(p.res, p.res_dtype, ri + e) : 0.0f;
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                if constexpr (EPI == XFTHIP_EPI_RESMUL) v[e] *= rv[e];
                if constexpr (EPI == XFTHIP_EPI_RESIDENTIAL) v[e] = v[e] + rv[e];
                if constexpr (EPI == XFTHIP_EPI_RESEXT) v[e] = fmaf(p.gamma, rv[e], v[e]);
            }
        }
        const size_t ci = (size_t)row * p.ldc + c;
        if (full && to.c_wide) {
            if (p.c_dtype == XFTHIP_F32) {
                const f32x4 o0 = {v[0], v[1], v[2], v[3]}, o1 = {v[4], v[5], v[6], v[7]};
                *(f32x4 *)((float *)p.C + ci) = o0;
                *(f32x4 *)((float *)p.C + ci + 4) = o1;
            } else {
                u32x4 o;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    o[e] = p.c_dtype == XFTHIP_BF16 ? f32x2_to_bf16(v[2 * e], v[2 * e + 1])
                                                    : (uint32_t)f32_to_fp16_bits(v[2 * e]) | ((uint32_t)f32_to_fp16_bits(v[2 * e + 1]) << 16);
                }
                *(u32x4 *)((uint16_t *)p.C + ci) = o;
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (c + e < col_end) store_from_f32(p.C, p.c_dtype, ci + e, v[e]);
        }
    }
    wave_sync();
}

// The launch of blocks of `rows` rows x 16 `tiles` columns: band_rows workgroups a unit of (band of row blocks, K part, column block), the units dealt out to the 8
// XCDs; a device-side row count may make up to a block a band and eight units more of a smaller number of row blocks
struct BlockGrid {
    int nblocks_n, nblocks_m, band, blocks;
};
template <bool DEVROWS>
static int block_grid(const SkinnyParams &p, int rows, int tiles, BlockGrid &g) {
    g.nblocks_n = (p.NTILES + tiles - 1) / tiles;
    // a group's row blocks: every weight may end in a partly filled one
    g.nblocks_m = (p.M + rows - 1) / rows + (p.group ? p.group_n : 0);
    const int parts = p.ksplit > 1 ? p.ksplit : 1;
    g.band = band_rows(g.nblocks_m, parts * g.nblocks_n);
    const int nbands = (g.nblocks_m + g.band - 1) / g.band;
    const long blocks = DEVROWS ? ((long)(g.nblocks_m + (g.nblocks_m + 7) / 8) * parts * g.nblocks_n + 64 + 7) / 8 * 8
                                : ((long)nbands * parts * g.nblocks_n + 7) / 8 * 8 * g.band;
    if (blocks > 0x7fffffffL) {
        set_error("qgemm_mfma: too many workgroups");
        return 2;
    }
    g.blocks = (int)blocks;
    return 0;
}

} // namespace
} // namespace xfthip
