// The gated delta-rule recurrence of layer plans: short convolutions, unit norms, decays and step sizes (delta_prepare), the
// walk over the tokens with the state in registers (delta_scan), both 16 tokens at a time in long segments (delta_chunk, delta_chunk_scan), the gated per-head norm behind it (delta_output).
// Everything between the projections' outputs and the output projection's input is fp32.
#include <algorithm>
#include <climits>
#include <type_traits>

#include "plan_dev.h"

namespace xfthip {

namespace {

template <bool BF16>
__device__ inline float ldb(const void *p, size_t i) {
    if constexpr (BF16) return bf16_to_f32(((const uint16_t *)p)[i]);
    else return ((const float *)p)[i];
}

struct PrepParams {
    StepView v;
    int below; // of the walk token by token: segments of as many tokens are taken in chunks
    DeltaBuffers b;
    const float *conv, *decay, *dt_bias;
    int H, KH, KD, VD, taps, ld, channels, beta_col, decay_col, gcols; // decay_col: one decay a head, in the row (or -1)
    float qscale;
};

// One wave a (token, head): its value channels, decay and step size, and (heads below KH) the query and key channels of
// key head `head`.  A channel is touched by one lane of one wave only, so that a sequence's single new token can shift the
// convolution's inputs in place; longer segments leave that to conv_tail_kernel.
template <bool BF16>
__global__ __launch_bounds__(256) void delta_prepare_kernel(PrepParams p) {
    const int lane = threadIdx.x & 63, t = blockIdx.x, head = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (head >= p.H) return;
    constexpr int DT = BF16 ? XFTHIP_BF16 : XFTHIP_F32;
    const int seg = p.v.tok_seg[t], pos = p.v.tok_pos[t];
    if (p.v.seg_len[seg] >= p.below) return;
    const int off = p.v.seg_off[seg], row = p.v.seg_row[seg];
    const bool alone = p.v.seg_len[seg] == 1;
    const int local = t - off;
    const size_t hist = (size_t)row * (p.taps - 1) * p.channels;
    auto conv = [&](int ch) {
        float acc = 0.0f;
        for (int j = 0; j < p.taps; ++j) {
            const int back = p.taps - 1 - j;
            if (pos < back) continue;
            const float in = local >= back ? load_as_f32(p.b.in, DT, (size_t)(t - back) * p.ld + ch)
                                           : load_as_f32(p.b.conv_state, DT, hist + (size_t)(p.taps - 1 + local - back) * p.channels + ch);
            acc = fmaf(p.conv[(size_t)ch * p.taps + j], in, acc);
        }
        if (alone) {
            for (int s = 0; s + 1 < p.taps - 1; ++s)
                store_from_f32(p.b.conv_state, DT, hist + (size_t)s * p.channels + ch, load_as_f32(p.b.conv_state, DT, hist + (size_t)(s + 1) * p.channels + ch));
            if (p.taps > 1)
                store_from_f32(p.b.conv_state, DT, hist + (size_t)(p.taps - 2) * p.channels + ch, load_as_f32(p.b.in, DT, (size_t)t * p.ld + ch));
        }
        return acc / (1.0f + expf(-acc));
    };
    if (head < p.KH) {
        float q[4], k[4], sq = 0.0f, sk = 0.0f, dot = 0.0f;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int c = i * 64 + lane;
            q[i] = k[i] = 0.0f;
            if (c < p.KD) {
                q[i] = conv(head * p.KD + c);
                k[i] = conv((p.KH + head) * p.KD + c);
            }
            sq = fmaf(q[i], q[i], sq), sk = fmaf(k[i], k[i], sk);
        }
        sq = 1.0f / sqrtf(wave_total(sq) + 1e-6f) * p.qscale;
        sk = 1.0f / sqrtf(wave_total(sk) + 1e-6f);
        const size_t at = ((size_t)t * p.KH + head) * p.KD;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int c = i * 64 + lane;
            q[i] *= sq, k[i] *= sk;
            dot = fmaf(q[i], k[i], dot);
            if (c < p.KD) p.b.q[at + c] = q[i], p.b.k[at + c] = k[i];
        }
        dot = wave_total(dot);
        if (lane == 0) p.b.qk[(size_t)t * p.KH + head] = dot;
    }
    for (int c = lane; c < p.VD; c += 64) p.b.v[((size_t)t * p.H + head) * p.VD + c] = conv(2 * p.KH * p.KD + head * p.VD + c);
    const float a = p.decay[head];
    if (p.decay_col >= 0) {
        const float x = load_as_f32(p.b.in, DT, (size_t)t * p.ld + p.decay_col + head) + p.dt_bias[head];
        if (lane == 0) p.b.g[(size_t)t * p.H + head] = expf(-a * (x > 20.0f ? x : log1pf(expf(x))));
    }
    for (int c = lane; c < p.KD && p.decay_col < 0; c += 64) {
        const float x = p.b.gates[(size_t)t * 2 * p.gcols + head * p.KD + c] + p.dt_bias[head * p.KD + c];
        const float sp = x > 20.0f ? x : log1pf(expf(x));
        p.b.g[((size_t)t * p.H + head) * p.KD + c] = expf(-a * sp);
    }
    if (lane == 0) p.b.beta[(size_t)t * p.H + head] = 1.0f / (1.0f + expf(-load_as_f32(p.b.in, DT, (size_t)t * p.ld + p.beta_col + head)));
}

// The same for the usual shapes (TAPS taps, head widths of at most 256): a wave walks TT consecutive tokens of one segment and
// head, two neighbouring channels a lane, the convolutions' last inputs in registers - every input is read once and every
// result leaves as a pair.  grid (token tiles of a segment, ceil(heads / 4), segments)
constexpr int kPrepTokens = 8;

template <bool BF16, int TAPS, int J> // J: turns of 128 channels that cover a head's width
__global__ __launch_bounds__(256) void delta_prepare_tiled_kernel(PrepParams p) {
    const int lane = threadIdx.x & 63, head = blockIdx.y * 4 + (threadIdx.x >> 6), seg = blockIdx.z;
    const int n = p.v.seg_len[seg], i0 = blockIdx.x * kPrepTokens;
    if (head >= p.H || i0 >= n || n >= p.below) return;
    const int off = p.v.seg_off[seg], row = p.v.seg_row[seg], start = p.v.seg_pos[seg];
    const int cnt = n - i0 < kPrepTokens ? n - i0 : kPrepTokens;
    const bool qk_head = head < p.KH;
    const size_t hist = (size_t)row * (TAPS - 1) * p.channels;
    const int vbase = 2 * p.KH * p.KD + head * p.VD;
    // input of channel pair c at local index i (negative: what earlier steps left; before the sequence's start: zero)
    auto input = [&](int c, int i) {
        if (start + i < 0) return make_float2(0.0f, 0.0f);
        return i >= 0 ? load2<BF16>(p.b.in, (size_t)(off + i) * p.ld + c) : load2<BF16>(p.b.conv_state, hist + (size_t)(TAPS - 1 + i) * p.channels + c);
    };
    struct Window {
        float2 w[TAPS]; // filter of either channel, tap by tap
        float2 x[TAPS > 1 ? TAPS - 1 : 1];
    };
    Window q[J], k[J], v[J];
    auto open = [&](Window &win, int c) {
#pragma unroll
        for (int t = 0; t < TAPS; ++t) win.w[t] = make_float2(p.conv[(size_t)c * TAPS + t], p.conv[(size_t)(c + 1) * TAPS + t]);
#pragma unroll
        for (int t = 0; t < TAPS - 1; ++t) win.x[t] = input(c, i0 - (TAPS - 1) + t);
    };
    auto advance = [&](Window &win, float2 in) { // silu of the filtered inputs; the window moves on by one token
        float2 a = make_float2(0.0f, 0.0f);
#pragma unroll
        for (int t = 0; t < TAPS - 1; ++t) a.x = fmaf(win.w[t].x, win.x[t].x, a.x), a.y = fmaf(win.w[t].y, win.x[t].y, a.y);
        a.x = fmaf(win.w[TAPS - 1].x, in.x, a.x), a.y = fmaf(win.w[TAPS - 1].y, in.y, a.y);
#pragma unroll
        for (int t = 0; t + 1 < TAPS - 1; ++t) win.x[t] = win.x[t + 1];
        if constexpr (TAPS > 1) win.x[TAPS - 2] = in;
        return make_float2(silu_of<BF16>(a.x), silu_of<BF16>(a.y));
    };
    float2 dtb[J];
#pragma unroll
    for (int j = 0; j < J; ++j) {
        const int c = j * 128 + lane * 2;
        if (qk_head && c < p.KD) open(q[j], head * p.KD + c), open(k[j], (p.KH + head) * p.KD + c);
        if (c < p.VD) open(v[j], vbase + c);
        dtb[j] = c < p.KD && p.decay_col < 0 ? *(const float2 *)(p.dt_bias + head * p.KD + c) : make_float2(0.0f, 0.0f);
    }
    const float decay = p.decay[head], head_dt = p.decay_col >= 0 ? p.dt_bias[head] : 0.0f;
    float2 nq[J], nk[J], nv[J], ng[J]; // the next token's values, requested a token ahead
    float nb = 0.0f, nd = 0.0f;
    auto request = [&](int i) {
        const int t = off + i;
        const size_t in_row = (size_t)t * p.ld;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int c = j * 128 + lane * 2;
            nq[j] = nk[j] = nv[j] = ng[j] = make_float2(0.0f, 0.0f);
            if (qk_head && c < p.KD) nq[j] = load2<BF16>(p.b.in, in_row + head * p.KD + c), nk[j] = load2<BF16>(p.b.in, in_row + (p.KH + head) * p.KD + c);
            if (c < p.VD) nv[j] = load2<BF16>(p.b.in, in_row + vbase + c);
            if (c < p.KD && p.decay_col < 0) ng[j] = *(const float2 *)(p.b.gates + (size_t)t * 2 * p.gcols + head * p.KD + c);
        }
        nb = ldb<BF16>(p.b.in, in_row + p.beta_col + head);
        if (p.decay_col >= 0) nd = ldb<BF16>(p.b.in, in_row + p.decay_col + head);
    };
    request(i0);
    for (int i = i0; i < i0 + cnt; ++i) {
        const int t = off + i;
        float2 xq[J], xk[J], xv[J], xg[J];
#pragma unroll
        for (int j = 0; j < J; ++j) xq[j] = nq[j], xk[j] = nk[j], xv[j] = nv[j], xg[j] = ng[j];
        const float bl = nb, dl = nd;
        if (i + 1 < i0 + cnt) request(i + 1);
        float sq = 0.0f, sk = 0.0f, dot = 0.0f;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int c = j * 128 + lane * 2;
            if (qk_head && c < p.KD) {
                xq[j] = advance(q[j], xq[j]), xk[j] = advance(k[j], xk[j]);
                sq = fmaf(xq[j].x, xq[j].x, fmaf(xq[j].y, xq[j].y, sq));
                sk = fmaf(xk[j].x, xk[j].x, fmaf(xk[j].y, xk[j].y, sk));
                dot = fmaf(xq[j].x, xk[j].x, fmaf(xq[j].y, xk[j].y, dot));
            }
            if (c < p.VD) *(float2 *)(p.b.v + ((size_t)t * p.H + head) * p.VD + c) = advance(v[j], xv[j]);
            if (c < p.KD && p.decay_col < 0) {
                *(float2 *)(p.b.g + ((size_t)t * p.H + head) * p.KD + c) = make_float2(exp_of<BF16>(-decay * softplus_of<BF16>(xg[j].x + dtb[j].x)),
                        exp_of<BF16>(-decay * softplus_of<BF16>(xg[j].y + dtb[j].y)));
            }
        }
        if (qk_head) { // (the same for the whole wave)
            sq = 1.0f / sqrtf(wave_total(sq) + 1e-6f) * p.qscale, sk = 1.0f / sqrtf(wave_total(sk) + 1e-6f);
            dot = wave_total(dot) * sq * sk;
            const size_t at = ((size_t)t * p.KH + head) * p.KD;
#pragma unroll
            for (int j = 0; j < J; ++j) {
                const int c = j * 128 + lane * 2;
                if (c < p.KD) {
                    *(float2 *)(p.b.q + at + c) = make_float2(xq[j].x * sq, xq[j].y * sq);
                    *(float2 *)(p.b.k + at + c) = make_float2(xk[j].x * sk, xk[j].y * sk);
                }
            }
            if (lane == 0) p.b.qk[(size_t)t * p.KH + head] = dot;
        }
        if (lane == 0) {
            p.b.beta[(size_t)t * p.H + head] = sigmoid_of<BF16>(bl);
            if (p.decay_col >= 0) p.b.g[(size_t)t * p.H + head] = exp_of<BF16>(-decay * softplus_of<BF16>(dl + head_dt));
        }
    }
    if (n == 1 && TAPS > 1) { // a single new token: nobody else reads these channels of the slot
        auto keep = [&](const Window &win, int c) {
#pragma unroll
            for (int t = 0; t < TAPS - 1; ++t) store2<BF16>(p.b.conv_state, hist + (size_t)t * p.channels + c, win.x[t]);
        };
#pragma unroll
        for (int j = 0; j < J; ++j) {
            const int c = j * 128 + lane * 2;
            if (qk_head && c < p.KD) keep(q[j], head * p.KD + c), keep(k[j], (p.KH + head) * p.KD + c);
            if (c < p.VD) keep(v[j], vbase + c);
        }
    }
}

struct TailParams {
    StepView v;
    const void *in;
    int ld, channels, taps;
    void *conv_state;
    int least;
};
// the last taps - 1 inputs of a segment of `least` tokens or more; one thread a channel
template <bool BF16>
__global__ __launch_bounds__(256) void conv_tail_kernel(TailParams p) {
    constexpr int DT = BF16 ? XFTHIP_BF16 : XFTHIP_F32;
    const int seg = blockIdx.y, n = p.v.seg_len[seg], ch = blockIdx.x * 256 + threadIdx.x;
    if (n < p.least || ch >= p.channels) return;
    const size_t hist = (size_t)p.v.seg_row[seg] * (p.taps - 1) * p.channels;
    const int off = p.v.seg_off[seg];
    for (int s = 0; s < p.taps - 1; ++s) { // ascending: slot s is read (as a later source) only by slots below it
        const int from = n - (p.taps - 1) + s;
        const float x = from >= 0 ? load_as_f32(p.in, DT, (size_t)(off + from) * p.ld + ch)
                                  : load_as_f32(p.conv_state, DT, hist + (size_t)(s + n) * p.channels + ch);
        store_from_f32(p.conv_state, DT, hist + (size_t)s * p.channels + ch, x);
    }
}

struct ScanParams {
    StepView v;
    DeltaBuffers b;
    int H, KH, VD, below; // (as above)
};

// The state's columns (value channels) do not interact.  L lanes hold C neighbouring columns, 4 RV key rows each (KD = 4 L RV).
// With S' = g S the step is a = S'^T k, b = S'^T q, u = beta (v - a), S = S' + k u^T, o = b + (q . k) u: both sums over the key
// rows run side by side and the read-out needs none of its own.  q, k, g of CT tokens are staged in LDS, the next CT on
// their way through registers.  grid (segments, heads, column groups of COLS).
// ONE: one decay a head, a scalar beside beta.
// What bounds it is the issue of instructions and, with few waves, their latency: four multiply-adds and less than one LDS read a state value.  So whatever
// else a token needs is kept small: the tokens of a full chunk are straight-line code whose LDS reads carry their offsets and go out a token ahead of
// their use; the read-outs' sums over the lanes, which nothing waits for, are left in LDS and added up for CT tokens at once, where a sum across the
// lanes was as many instructions as the one that the chain needs; the last half of the column groups walk the segments backwards, so that an XCD and a CU
// (which take every 8th and every 256th workgroup) get long and short ones.  16 heads of 128 x 128, before and after: two prompts of 3000 tokens
// at most 690 / 600 us, four of 940 to 1500 420 / 350, eight of 800 at most 404 / 272, 16 of 400 346 / 230, 24 of 500 600 / 520.  One of 2000 tokens: 32 heads 430 /
// 377, 4 heads 408 / 343, 16 heads of 64 x 64 401 / 325, of 256 x 256 716 / 637; with one decay a head, 32 heads 409 / 350; one of 8 tokens 4.1 / 4.1.
// (KD = 128 as 32 lanes x 4 rows x 2 columns, half the LDS reads: 510 us for 2048 tokens against 440 as 16 x 8 x 1.)
template <int L, int RV, int C, bool ONE>
__global__ __launch_bounds__(256) void delta_scan_kernel(ScanParams p) {
    constexpr int KD = 4 * L * RV, GROUPS = 256 / L, COLS = GROUPS * C, CT = 8;
    constexpr int CHUNK4 = CT * KD / 4; // float4 of one array and chunk
    constexpr int ARRAYS = ONE ? 2 : 3, SCALARS = ONE ? 3 : 2; // q, k(, g); beta, q . k(, g)
    constexpr int PER = (ARRAYS * CHUNK4 + 255) / 256, PERV = (CT * COLS + 255) / 256;
    __shared__ float lds[2][ARRAYS * CT * KD];
    __shared__ float vlds[2][CT * COLS];
    __shared__ float sc[2][SCALARS * CT];
    __shared__ f32x4 sums[CT * COLS * L / 4]; // the lanes' parts of the read-outs: [token][c][column group][lane]
    const int seg = 2 * blockIdx.z < gridDim.z ? blockIdx.x : gridDim.x - 1 - blockIdx.x, head = blockIdx.y, kvh = head / (p.H / p.KH);
    const int n = p.v.seg_len[seg], off = p.v.seg_off[seg];
    if (n >= p.below) return;
    const int li = threadIdx.x % L, lc = threadIdx.x / L * C;
    const int col0 = blockIdx.z * COLS, col = col0 + lc;
    const bool own = col < p.VD; // (VD is a multiple of 32: C neighbouring columns are in it or not together)
    float *state = p.b.state + (((size_t)p.v.seg_row[seg] * p.H + head) * p.VD + (own ? col : 0)) * KD + 4 * li;
    f32x4 s[C][RV];
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int r = 0; r < RV; ++r) s[c][r] = p.v.seg_pos[seg] > 0 ? *(const f32x4 *)(state + c * KD + r * 4 * L) : f32x4 {0.f, 0.f, 0.f, 0.f};

    f32x4 stage[PER];
    float vstage[PERV], cstage = 0.0f;
    // (threads without a part fetch the last one: a load under a condition would be waited for before the next one goes out)
    auto fetch = [&](int c0) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int part = i * 256 + (int)threadIdx.x, e = part < ARRAYS * CHUNK4 ? part : ARRAYS * CHUNK4 - 1;
            const int arr = e / CHUNK4, r = e % CHUNK4, tok = r / (KD / 4), d = (r % (KD / 4)) * 4;
            const int t = off + (c0 + tok < n ? c0 + tok : n - 1);
            const float *src = arr == 2 ? p.b.g + ((size_t)t * p.H + head) * KD : (arr ? p.b.k : p.b.q) + ((size_t)t * p.KH + kvh) * KD;
            stage[i] = *(const f32x4 *)(src + d);
        }
#pragma unroll
        for (int i = 0; i < PERV; ++i) {
            const int part = i * 256 + (int)threadIdx.x, e = part < CT * COLS ? part : CT * COLS - 1, tok = e / COLS, c = col0 + e % COLS;
            const int t = off + (c0 + tok < n ? c0 + tok : n - 1);
            vstage[i] = p.b.v[((size_t)t * p.H + head) * p.VD + (c < p.VD ? c : p.VD - 1)];
        }
        const int tok = threadIdx.x % CT, t = off + (c0 + tok < n ? c0 + tok : n - 1);
        const float *scalar = threadIdx.x < CT ? p.b.beta + (size_t)t * p.H + head : threadIdx.x < 2 * CT || !ONE ? p.b.qk + (size_t)t * p.KH + kvh : p.b.g + (size_t)t * p.H + head;
        cstage = *scalar;
    };
    auto stash = [&](int buf) {
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int e = i * 256 + threadIdx.x;
            if (e < ARRAYS * CHUNK4) *(f32x4 *)(&lds[buf][4 * e]) = stage[i];
        }
#pragma unroll
        for (int i = 0; i < PERV; ++i) {
            const int e = i * 256 + threadIdx.x;
            if (e < CT * COLS) vlds[buf][e] = vstage[i];
        }
        if (threadIdx.x < SCALARS * CT) sc[buf][threadIdx.x] = cstage;
    };
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
        for (int r = 0; r < RV; ++r) arrived(s[c][r]);
    fetch(0);
    stash(0);
    __syncthreads();
    int buf = 0;
    for (int c0 = 0; c0 < n; c0 += CT, buf ^= 1) {
        const int m = n - c0 < CT ? n - c0 : CT;
        if (c0 + CT < n) fetch(c0 + CT);
        const float *lq = lds[buf] + 4 * li;
        float *part = (float *)sums + threadIdx.x;
        struct Operands {
            f32x4 q[RV], k[RV], g[ONE ? 1 : RV];
            float v[C], beta, qk, fade;
        };
        auto read = [&](int i) {
            const float *q = lq + i * KD, *k = q + CT * KD, *g = k + CT * KD;
            Operands x;
#pragma unroll
            for (int r = 0; r < RV; ++r) {
                x.q[r] = *(const f32x4 *)(q + r * 4 * L), x.k[r] = *(const f32x4 *)(k + r * 4 * L);
                if constexpr (!ONE) x.g[r] = *(const f32x4 *)(g + r * 4 * L);
            }
#pragma unroll
            for (int c = 0; c < C; ++c) x.v[c] = vlds[buf][i * COLS + lc + c];
            x.beta = sc[buf][i], x.qk = sc[buf][CT + i];
            if constexpr (ONE) x.fade = sc[buf][2 * CT + i];
            return x;
        };
        // the operands of the next token are on their way from LDS while this one's sums go round
        auto token = [&](const Operands &x, int i) {
            float a[C], b[C];
#pragma unroll
            for (int c = 0; c < C; ++c) {
                a[c] = b[c] = 0.0f;
#pragma unroll
                for (int r = 0; r < RV; ++r)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        if constexpr (ONE) s[c][r][e] *= x.fade;
                        else s[c][r][e] *= x.g[r][e];
                        a[c] = fmaf(x.k[r][e], s[c][r][e], a[c]), b[c] = fmaf(x.q[r][e], s[c][r][e], b[c]);
                    }
            }
#pragma unroll
            for (int c = 0; c < C; ++c) a[c] = group_sum<L>(a[c]);
#pragma unroll
            for (int c = 0; c < C; ++c) {
                const float u = x.beta * (x.v[c] - a[c]);
#pragma unroll
                for (int r = 0; r < RV; ++r)
#pragma unroll
                    for (int e = 0; e < 4; ++e) s[c][r][e] = fmaf(x.k[r][e], u, s[c][r][e]);
                const float with = fmaf(x.qk, u, b[c]);
                part[(i * C + c) * 256] = li == 0 ? with : b[c];
            }
        };
        Operands even = read(0), odd;
        if (m == CT) {
#pragma unroll
            for (int i = 0; i < CT; i += 2) {
                odd = read(i + 1);
                __builtin_amdgcn_sched_barrier(0);
                token(even, i);
                __builtin_amdgcn_sched_barrier(0);
                if (i + 2 < CT) even = read(i + 2);
                __builtin_amdgcn_sched_barrier(0);
                token(odd, i + 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            for (int i = 0; i < m; ++i) {
                token(even, i);
                even = read(i + 1 < m ? i + 1 : i);
            }
        }
        if (c0 + CT < n) stash(buf ^ 1); // (that buffer was last read in front of the barrier one chunk ago)
        // The read-outs of a wave's own columns: written and read by the same wave, whose LDS accesses keep their order.  64 / L column groups a wave.
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        constexpr int WG = 64 / L, OUTS = CT * C * WG;
#pragma unroll
        for (int o0 = 0; o0 < OUTS; o0 += 64) {
            const int o = o0 + (threadIdx.x & 63), i = o / (C * WG), at = o % (C * WG), c = at % C, gr = (threadIdx.x >> 6) * WG + at / C;
            if (i >= m) continue;
            const f32x4 *x = sums + ((i * C + c) * GROUPS + gr) * (L / 4);
            f32x4 y = x[(o >> 2) % (L / 4)]; // (lanes begin at different quarters: at the same one they would share banks)
#pragma unroll
            for (int r = 1; r < L / 4; ++r) y += x[(r + (o >> 2)) % (L / 4)];
            const int vc = col0 + gr * C + c;
            if (vc < p.VD) p.b.o[((size_t)(off + c0 + i) * p.H + head) * p.VD + vc] = (y[0] + y[1]) + (y[2] + y[3]);
        }
        __syncthreads();
    }
    if (own) {
#pragma unroll
        for (int c = 0; c < C; ++c)
#pragma unroll
            for (int r = 0; r < RV; ++r) *(f32x4 *)(state + c * KD + r * 4 * L) = s[c][r];
    }
}

// ---- segments of many tokens, kChunk at a time ----------------------------------------------------
// Within a chunk, with G_t the product of the decays up to token t and G_t / G_s that of those behind s (always multiplied out, never divided):
//   a_t = (G_t k_t)^T S_0 + sum_{s < t} A_ts u_s,   A_ts = k_t^T (G_t / G_s) k_s,   u_t = beta_t (v_t - a_t)
//   o_t = (G_t q_t)^T S_0 + sum_{s <= t} B_ts u_s,  B_ts = q_t^T (G_t / G_s) k_s
//   S   = G_16 S_0 + sum_s (G_16 / G_s) k_s u_s^T
// so u = U (v - W S_0) with W = G k and U = (1 + beta A)^-1 beta, a triangular matrix whose entries are bounded by one (products of contractions): what a chunk does to
// the state's columns are products of matrices that no column has a part in.
// Record of a (chunk, head) for the scan: W [16][KD] | G q [16][KD] | (G_16 / G_s) k_s as [KD][16] | G_16 [KD] | U [16][16] | B [16][16]
constexpr int kChunk = 16;
__host__ __device__ constexpr size_t chunk_floats(int KD) { return (size_t)(3 * kChunk + 1) * KD + 2 * kChunk * kChunk; }
// records in front of a segment's: ceil(n / 16) of every segment fit in floor((off + n) / 16) - floor(off / 16) + 1
__device__ inline size_t chunk_of(int off, int seg) { return (size_t)(off / kChunk + seg); }
// the segments of a launch
constexpr int kChunkSegs = 128;
struct ChunkSegs {
    int seg[kChunkSegs];
};

// In place of delta_prepare for such segments: convolutions, norms and decays of a (chunk, head) by a workgroup of its own, two neighbouring channels of q, k, v or the decays a
// thread, and what the scan needs of them.  Tokens past the segment's end have no keys, queries and step sizes.  A and B: thread (s, 1/16 of the key dims) carries k_s on from token to token,
// 16 lanes add up.  Bound by the round trips of a workgroup, of which four share a CU (112 registers; LDS would take five; 4 prompts of 1000 to 1500 tokens, 16 heads of 128 x 128: 110 us for 270 MB; delta_prepare, which
// leaves the products to the scan, 85).
template <int KD, bool ONE, bool BF16>
__global__ __launch_bounds__(256) void delta_chunk_kernel(PrepParams p, ChunkSegs segs) {
    constexpr int J = KD / 64, N = kChunk * KD / 4 / 256, P = KD + 4, SIZE = kChunk * P; // (rows of P: lanes that read a column of rows are on banks of their own)
    __shared__ __align__(16) float q[SIZE], k[SIZE], g[SIZE], A[kChunk * kChunk], B[kChunk * kChunk], beta[kChunk], one[kChunk];
    const int tid = threadIdx.x, head = blockIdx.y, seg = segs.seg[blockIdx.z], H = p.H, kvh = head / (H / p.KH), c0 = blockIdx.x * kChunk;
    const int n = p.v.seg_len[seg], off = p.v.seg_off[seg], start = p.v.seg_pos[seg], taps = p.taps;
    if (c0 >= n) return;
    const size_t hist = (size_t)p.v.seg_row[seg] * (taps - 1) * p.channels;
    const int cnt = n - c0 < kChunk ? n - c0 : kChunk;
    const float decay = p.decay[head];
    constexpr int W = KD / 2;
    for (int w = tid; w < (ONE ? 2 : 3) * W + p.VD / 2; w += 256) {
        if (!ONE && w >= 2 * W + p.VD / 2) {
            const int d = 2 * (w - 2 * W - p.VD / 2);
            const float2 dt = *(const float2 *)(p.dt_bias + head * KD + d);
            float2 x[kChunk];
#pragma unroll
            for (int i = 0; i < kChunk; ++i) x[i] = *(const float2 *)(p.b.gates + (size_t)(off + c0 + (i < cnt ? i : 0)) * 2 * p.gcols + head * KD + d);
#pragma unroll
            for (int i = 0; i < kChunk; ++i)
                *(float2 *)(g + i * P + d) = i < cnt ? make_float2(exp_of<BF16>(-decay * softplus_of<BF16>(x[i].x + dt.x)), exp_of<BF16>(-decay * softplus_of<BF16>(x[i].y + dt.y)))
                                                     : make_float2(1.0f, 1.0f);
            continue;
        }
        const int c = w < W ? kvh * KD + 2 * w : w < 2 * W ? (p.KH + kvh) * KD + 2 * (w - W) : 2 * p.KH * KD + head * p.VD + 2 * (w - 2 * W);
        float2 f[4], x[kChunk + 3]; // the last of four taps; inputs from three in front of the chunk on: of earlier steps what they left, before the sequence's start zero
#pragma unroll
        for (int j = 0; j < 4; ++j)
            f[j] = j >= 4 - taps ? make_float2(p.conv[(size_t)c * taps + j - (4 - taps)], p.conv[(size_t)(c + 1) * taps + j - (4 - taps)]) : make_float2(0.0f, 0.0f);
#pragma unroll
        for (int j = 0; j < kChunk + 3; ++j) {
            const int i = c0 + j - 3;
            x[j] = make_float2(0.0f, 0.0f);
            if (j >= 3) x[j] = load2<BF16>(p.b.in, (size_t)(off + (j - 3 < cnt ? i : c0)) * p.ld + c);
            else if (j >= 4 - taps && start + i >= 0)
                x[j] = i >= 0 ? load2<BF16>(p.b.in, (size_t)(off + i) * p.ld + c) : load2<BF16>(p.b.conv_state, hist + (size_t)(taps - 1 + i) * p.channels + c);
        }
#pragma unroll
        for (int i = 0; i < kChunk; ++i) {
            float2 a = make_float2(0.0f, 0.0f);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (j >= 4 - taps) a.x = fmaf(f[j].x, x[i + j].x, a.x), a.y = fmaf(f[j].y, x[i + j].y, a.y);
            a = i < cnt ? make_float2(silu_of<BF16>(a.x), silu_of<BF16>(a.y)) : make_float2(0.0f, 0.0f);
            if (w < 2 * W) *(float2 *)((w < W ? q + 2 * w : k + 2 * (w - W)) + i * P) = a;
            else if (i < cnt) *(float2 *)(p.b.v + ((size_t)(off + c0 + i) * H + head) * p.VD + 2 * (w - 2 * W)) = a;
        }
    }
    if (tid < kChunk) {
        const size_t t = (size_t)(off + c0 + (tid < cnt ? tid : 0)) * p.ld;
        beta[tid] = tid < cnt ? sigmoid_of<BF16>(ldb<BF16>(p.b.in, t + p.beta_col + head)) : 0.0f;
        if constexpr (ONE) one[tid] = tid < cnt ? exp_of<BF16>(-decay * softplus_of<BF16>(ldb<BF16>(p.b.in, t + p.decay_col + head) + p.dt_bias[head])) : 1.0f;
    }
    __syncthreads();
    {
        f32x4 x[J], y[J];
        float *qt = q + (tid >> 4) * P + 4 * (tid & 15), *kt = k + (tid >> 4) * P + 4 * (tid & 15), sq = 0.0f, sk = 0.0f;
#pragma unroll
        for (int j = 0; j < J; ++j) {
            x[j] = *(const f32x4 *)(qt + 64 * j), y[j] = *(const f32x4 *)(kt + 64 * j);
#pragma unroll
            for (int e = 0; e < 4; ++e) sq = fmaf(x[j][e], x[j][e], sq), sk = fmaf(y[j][e], y[j][e], sk);
        }
        sq = 1.0f / sqrtf(group_sum<16>(sq) + 1e-6f) * p.qscale, sk = 1.0f / sqrtf(group_sum<16>(sk) + 1e-6f);
#pragma unroll
        for (int j = 0; j < J; ++j) {
#pragma unroll
            for (int e = 0; e < 4; ++e) x[j][e] *= sq, y[j][e] *= sk;
            *(f32x4 *)(qt + 64 * j) = x[j], *(f32x4 *)(kt + 64 * j) = y[j];
        }
    }
    A[tid] = B[tid] = 0.0f;
    __syncthreads();
    float *rec = p.b.chunks + ((chunk_of(off, seg) + blockIdx.x) * H + head) * chunk_floats(KD);
    {
        const int s = tid >> 4, part = 4 * (tid & 15);
        f32x4 r[J];
#pragma unroll
        for (int j = 0; j < J; ++j) r[j] = f32x4 {0.f, 0.f, 0.f, 0.f};
        for (int t0 = s & ~3; t0 < kChunk; t0 += 4) { // (from the wave's first key on)
            float x[4], y[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int t = t0 + i;
                x[i] = y[i] = 0.0f;
#pragma unroll
                for (int j = 0; j < J; ++j) {
                    const int at = t * P + part + 64 * j;
                    const f32x4 kt = *(const f32x4 *)(k + at), qt = *(const f32x4 *)(q + at);
                    f32x4 gt;
                    if constexpr (ONE) gt = f32x4 {one[t], one[t], one[t], one[t]};
                    else gt = *(const f32x4 *)(g + at);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        r[j][e] = t == s ? kt[e] : t > s ? r[j][e] * gt[e] : 0.0f;
                        x[i] = fmaf(kt[e], r[j][e], x[i]), y[i] = fmaf(qt[e], r[j][e], y[i]);
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = group_sum<16>(x[i]), y[i] = group_sum<16>(y[i]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (part == 0 && t0 + i > s) A[(t0 + i) * kChunk + s] = x[i];
                if (part == 0 && t0 + i >= s) B[(t0 + i) * kChunk + s] = y[i];
            }
        }
    }
    // a thread's channel of the keys or of the queries, in place: times the decays' products from the front, and from the back where the decays lie
    constexpr int M = KD > 128 ? 2 : 1;
    float x[M][kChunk], y[M][kChunk];
    auto channel = [&](int m) { return KD > 128 ? tid : tid % KD; };
    auto keys = [&](int m) { return KD > 128 ? m == 0 : tid < KD; };
    const bool mine = tid < 2 * KD;
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int t = 0; t < kChunk && mine; ++t) x[m][t] = (keys(m) ? k : q)[t * P + channel(m)], y[m][t] = ONE ? one[t] : g[t * P + channel(m)];
    __syncthreads();
#pragma unroll
    for (int m = 0; m < M && mine; ++m) {
        const int d = channel(m);
        float G = 1.0f;
        if (keys(m)) {
#pragma unroll
            for (int t = kChunk - 1; t >= 0; --t) g[t * P + d] = G * x[m][t], G *= y[m][t];
            rec[3 * kChunk * KD + d] = G, G = 1.0f;
#pragma unroll
            for (int t = 0; t < kChunk; ++t) G *= y[m][t], k[t * P + d] = G * x[m][t];
        } else {
#pragma unroll
            for (int t = 0; t < kChunk; ++t) G *= y[m][t], q[t * P + d] = G * x[m][t];
        }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const int e = i * 256 + tid, at = (e & 15) * P + (e >> 6 << 4 | (e >> 2 & 12)); // token, four key rows
        *(f32x4 *)(rec + 4 * e) = *(const f32x4 *)(k + at), *(f32x4 *)(rec + kChunk * KD + 4 * e) = *(const f32x4 *)(q + at);
        const float *from = g + 4 * (e & 3) * P + (e >> 2); // four tokens, key row
        *(f32x4 *)(rec + 2 * kChunk * KD + 4 * e) = f32x4 {from[0], from[P], from[2 * P], from[3 * P]};
    }
    rec += (3 * kChunk + 1) * KD;
    rec[kChunk * kChunk + tid] = B[tid];
    if (tid >= 256 - kChunk) { // column s of -U, row by row: what token t leaves is taken from all behind it at once
        const int s = tid - (256 - kChunk);
        float u[kChunk];
#pragma unroll
        for (int t = 0; t < kChunk; ++t) u[t] = t == s ? -1.0f : 0.0f;
#pragma unroll
        for (int t = 0; t < kChunk; ++t) {
            u[t] = t < s ? 0.0f : beta[t] * u[t];
#pragma unroll
            for (int r = t + 1; r < kChunk; ++r) u[r] = fmaf(-A[r * kChunk + t], u[t], u[r]);
        }
#pragma unroll
        for (int t = 0; t < kChunk; ++t) rec[t * kChunk + s] = u[t];
    }
}

// A wave holds 16 columns of a head's state as accumulators of 16 x 16 x 4 fp32 MFMAs, key row 16 i + 4 g + r in register r of tile i (g = lane / 16): with key rows dealt to the MFMAs'
// k slots alike they are the operand of W S_0 and (G q) S_0 as they lie, as are the results, rows of tokens, of the products with U, B and the keys: nothing moves between lanes.
// NW waves share the key rows and add up their parts of W S_0 and (G q) S_0 through LDS; one more makes the outputs, off the chain from state to state.  Wave 0 takes v from its part, the
// records hold -U.  C tiles of 16 columns a wave.  Every operand is requested two chunks ahead, behind its last use.
// Bound by the chain: products, barrier, sums, the product with U and the check of it, the state's products, about 2000 clocks a chunk of which the MFMAs fill 930, and by the MFMAs where a SIMD
// has several waves of it; the scan above takes 600 clocks a token.  prepare and scan, before and after, us: 16 heads of 128 x 128, one prompt of 1500
// tokens 296 / 124, two of 3000 646 / 300, 4 of 1000 to 1500 429 / 264, 8 of 800 416 / 308, 16 of 400 399 / 314, one of 32 31 / 22; 16 of 64 x 64, 8 of 800 224 / 142; 8 of 256 x 256, 2 of
// 3000 1038 / 431, 16 of 400 816 / 441; with one decay a head, 32 of 128 x 128, 2 of 3000 784 / 468, 16 of 400 603 / 526.
// A wave for all key rows: 213 us for the prompt of 1500, two 103, four 82 (85 with two sums of every product, for as small an error as the walk token by token has).  With the stores of a last, ragged chunk in the loop every wait was one for the stores before, too: 100.
template <int KD, int NW, int C>
__global__ __launch_bounds__(64 * NW + 64, KD / NW == 32 && C == 1 ? 4 : 2) void delta_chunk_scan_kernel(ScanParams p, ChunkSegs segs) {
    constexpr int I = KD / 16 / NW, SETS = 2;
    __shared__ f32x4 parts[2][NW][2][C][64];
    // (segments of one place are handed to one XCD in turn, whose share should be long and short ones)
    const int seg = segs.seg[(blockIdx.x + blockIdx.y + (blockIdx.y >> 1) + (blockIdx.y >> 2)) % gridDim.x], head = blockIdx.y, lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int g = lane >> 4, c = lane & 15, row0 = wave * 16 * I;
    const int n = p.v.seg_len[seg], off = p.v.seg_off[seg], last = (n - 1) / kChunk;
    // addresses: scalar ones that move with the chunks, and these of a lane (in bytes), which do not
    const char *records = (const char *)(p.b.chunks + (chunk_of(off, seg) * p.H + head) * chunk_floats(KD));
    const size_t next = (size_t)p.H * chunk_floats(KD) * 4, first = ((size_t)off * p.H + head) * p.VD + blockIdx.z * 16 * C;
    const uint32_t row = (uint32_t)p.H * p.VD * 4, at_u = (c * kChunk + 4 * g) * 4;
    uint32_t token[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) token[r] = (4 * g + r) * row;
    auto load = [](const char *base, uint32_t at) { return *(const f32x4 *)(base + at); };
    auto times = [&](const f32x4 m, const f32x4 y, f32x4 d) {
#pragma unroll
        for (int e = 0; e < 4; ++e) d = __builtin_amdgcn_mfma_f32_16x16x4f32(m[e], y[e], d, 0, 0, 0);
        return d;
    };
    auto finite = [&](const f32x4 (&y)[C]) {
        float z = 0.0f;
#pragma unroll
        for (int t = 0; t < C; ++t) z += (y[t][0] * 0.0f + y[t][1] * 0.0f) + (y[t][2] * 0.0f + y[t][3] * 0.0f);
        return __builtin_amdgcn_ballot_w64(!(z == 0.0f)) == 0;
    };
    // what a token must not see of later ones, though their factors are zero: row t with the values up to it alone
    auto times_row_by_row = [&](const f32x4 m, const f32x4 y, const f32x4 d) {
        f32x4 out = d;
#pragma unroll 1
        for (int t = 0; t < kChunk; ++t) {
            f32x4 z;
#pragma unroll
            for (int e = 0; e < 4; ++e) z[e] = 4 * g + e <= t ? y[e] : 0.0f;
            z = times(m, z, d);
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (4 * g + e == t) out[e] = z[e];
        }
        return out;
    };
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    auto record = [&](int chunk) { return records + (chunk < last ? chunk : last) * next; }; // (behind the last: the last again)
    // every wave's u from the parts of W S_0 - v; sound: nothing infinite in it, nor in what it was made of
    auto solve = [&](const f32x4 m, int chunk, int buf, f32x4 (&u)[C]) {
        f32x4 r[C];
#pragma unroll
        for (int t = 0; t < C; ++t) {
            r[t] = parts[buf][0][0][t][lane], u[t] = zero;
#pragma unroll
            for (int w = 1; w < NW; ++w) r[t] += parts[buf][w][0][t][lane];
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int t = 0; t < C; ++t) u[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(m[e], r[t][e], u[t], 0, 0, 0);
        const bool sound = finite(u);
        if (!sound) {
#pragma unroll
            for (int t = 0; t < C; ++t) {
                u[t] = times_row_by_row(m, r[t], zero);
#pragma unroll
                for (int e = 0; e < 4; ++e) u[t][e] = 4 * g + e < n - chunk * kChunk ? u[t][e] : 0.0f;
            }
        }
        return sound;
    };
    // (a buffer's readers of two chunks ago have passed the barrier of one chunk ago)
    auto meet = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    int chunk = 0;
    if (wave == NW) {
        // the read-outs
        struct Outs {
            f32x4 u, b;
        };
        Outs set[SETS];
        auto fetch = [&](Outs &o, int chunk) {
            const char *rec = record(chunk) + (3 * kChunk + 1) * KD * 4;
            o.u = load(rec, at_u), o.b = load(rec + kChunk * kChunk * 4, at_u);
        };
        // (the last chunk's stores, of which some may be left out, have a place of their own: the count of a wait in the loop would have to do without them and be that of a wait
        // for the stores before, too)
        auto step = [&](Outs &o, int chunk, int buf, auto whole) {
            f32x4 u[C];
            meet();
            const bool sound = solve(o.u, chunk, buf, u);
            char *out = (char *)(p.b.o + first) + (size_t)chunk * kChunk * row;
#pragma unroll
            for (int t = 0; t < C; ++t) {
                f32x4 b = parts[buf][0][1][t][lane];
#pragma unroll
                for (int w = 1; w < NW; ++w) b += parts[buf][w][1][t][lane];
                b = sound ? times(o.b, u[t], b) : times_row_by_row(o.b, u[t], b);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (whole() || 4 * g + e < n - chunk * kChunk) *(float *)(out + 64 * t + (token[e] + 4 * c)) = b[e];
            }
            __builtin_amdgcn_sched_barrier(0);
            fetch(o, chunk + SETS);
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int i = 0; i < SETS; ++i) fetch(set[i], i);
        for (; chunk + SETS <= last; chunk += SETS)
#pragma unroll
            for (int i = 0; i < SETS; ++i) step(set[i], chunk + i, (chunk + i) & 1, std::true_type());
#pragma unroll
        for (int i = 0; i < SETS; ++i) {
            if (chunk + i == last) step(set[i], last, last & 1, std::false_type());
            else if (chunk + i < last) step(set[i], chunk + i, (chunk + i) & 1, std::true_type());
        }
        return;
    }
    const uint32_t at_w = row0 * 64 + lane * 16, at_x = ((row0 + c) * kChunk + 4 * g) * 4, at_fade = (row0 + 4 * g) * 4;
    float *state = p.b.state + (((size_t)p.v.seg_row[seg] * p.H + head) * p.VD + blockIdx.z * 16 * C + c) * KD + row0 + 4 * g;
    f32x4 s[C][I];
#pragma unroll
    for (int t = 0; t < C; ++t)
#pragma unroll
        for (int i = 0; i < I; ++i) s[t][i] = p.v.seg_pos[seg] > 0 ? *(const f32x4 *)(state + t * 16 * KD + 16 * i) : zero;
    struct Operands {
        f32x4 w[I], q[I], x[I], fade[I], u, v[C];
    };
    Operands set[SETS];
#pragma unroll
    for (int i = 0; i < SETS; ++i)
#pragma unroll
        for (int t = 0; t < C; ++t) set[i].v[t] = zero; // (one wave takes the values from its part)
    auto fetch_w = [&](Operands &o, int chunk) {
        const char *rec = record(chunk);
#pragma unroll
        for (int i = 0; i < I; ++i) o.w[i] = load(rec + 1024 * i, at_w), o.q[i] = load(rec + kChunk * KD * 4 + 1024 * i, at_w);
        if (wave != 0) return;
        const int here = chunk < last ? chunk : last, most = n - 1 - here * kChunk;
        const char *v = (const char *)(p.b.v + first) + (size_t)here * kChunk * row;
        const uint32_t end = (most < kChunk - 1 ? most : kChunk - 1) * row; // (tokens behind it: the last one's, which count for nothing)
#pragma unroll
        for (int t = 0; t < C; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) o.v[t][r] = *(const float *)(v + 64 * t + ((token[r] < end ? token[r] : end) + 4 * c));
    };
    auto fetch_x = [&](Operands &o, int chunk) {
        const char *rec = record(chunk) + 2 * kChunk * KD * 4;
        o.u = load(rec + (kChunk + 1) * KD * 4, at_u);
#pragma unroll
        for (int i = 0; i < I; ++i) o.fade[i] = load(rec + kChunk * KD * 4 + 64 * i, at_fade);
#pragma unroll
        for (int i = 0; i < I; ++i) o.x[i] = load(rec + kChunk * 64 * i, at_x);
    };
#pragma unroll
    for (int t = 0; t < C; ++t)
#pragma unroll
        for (int i = 0; i < I; ++i) arrived(s[t][i]);
    auto step = [&](Operands &o, int chunk, int buf) {
        f32x4 a[C][2], b[C][2], u[C];
#pragma unroll
        for (int t = 0; t < C; ++t) a[t][0] = a[t][1] = b[t][0] = b[t][1] = zero;
#pragma unroll
        for (int i = 0; i < I; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int t = 0; t < C; ++t)
                    a[t][i & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.w[i][e], s[t][i][e], a[t][i & 1], 0, 0, 0),
                    b[t][i & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.q[i][e], s[t][i][e], b[t][i & 1], 0, 0, 0);
#pragma unroll
        for (int t = 0; t < C; ++t) parts[buf][wave][0][t][lane] = (a[t][0] + a[t][1]) - o.v[t], parts[buf][wave][1][t][lane] = b[t][0] + b[t][1];
        __builtin_amdgcn_sched_barrier(0);
        fetch_w(o, chunk + SETS);
        meet();
        solve(o.u, chunk, buf, u);
#pragma unroll
        for (int t = 0; t < C; ++t)
#pragma unroll
            for (int i = 0; i < I; ++i) s[t][i] = s[t][i] * o.fade[i];
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < I; ++i)
#pragma unroll
                for (int t = 0; t < C; ++t) s[t][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(o.x[i][e], u[t][e], s[t][i], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        fetch_x(o, chunk + SETS);
        __builtin_amdgcn_sched_barrier(0);
    };
#pragma unroll
    for (int i = 0; i < SETS; ++i) fetch_w(set[i], i), fetch_x(set[i], i);
    for (; chunk + SETS - 1 <= last; chunk += SETS)
#pragma unroll
        for (int i = 0; i < SETS; ++i) step(set[i], chunk + i, (chunk + i) & 1);
#pragma unroll
    for (int i = 0; i + 1 < SETS; ++i)
        if (chunk + i <= last) step(set[i], chunk + i, (chunk + i) & 1);
#pragma unroll
    for (int t = 0; t < C; ++t)
#pragma unroll
        for (int i = 0; i < I; ++i) *(f32x4 *)(state + t * 16 * KD + 16 * i) = s[t][i];
}

// The same step for segments of one token: nothing to stage, the kernel is a read and a write of the state.
template <int L, bool ONE>
__global__ __launch_bounds__(256) void delta_step_kernel(ScanParams p) {
    constexpr int KD = 8 * L, COLS = 256 / L;
    const int seg = blockIdx.x, head = blockIdx.y, kvh = head / (p.H / p.KH), t = p.v.seg_off[seg];
    const int li = threadIdx.x % L, col = blockIdx.z * COLS + threadIdx.x / L;
    if (col >= p.VD || p.v.seg_len[seg] >= p.below) return; // (whole groups of L lanes)
    float *state = p.b.state + (((size_t)p.v.seg_row[seg] * p.H + head) * p.VD + col) * KD;
    f32x4 s0 = *(const f32x4 *)(state + 4 * li), s1 = *(const f32x4 *)(state + 4 * (L + li));
    const float *q = p.b.q + ((size_t)t * p.KH + kvh) * KD + 4 * li, *k = p.b.k + ((size_t)t * p.KH + kvh) * KD + 4 * li;
    f32x4 g0, g1;
    if constexpr (ONE) {
        const float fade = p.b.g[(size_t)t * p.H + head];
        g0 = g1 = f32x4 {fade, fade, fade, fade};
    } else {
        const float *g = p.b.g + ((size_t)t * p.H + head) * KD + 4 * li;
        g0 = *(const f32x4 *)g, g1 = *(const f32x4 *)(g + 4 * L);
    }
    const f32x4 q0 = *(const f32x4 *)q, q1 = *(const f32x4 *)(q + 4 * L), k0 = *(const f32x4 *)k, k1 = *(const f32x4 *)(k + 4 * L);
    const float v = p.b.v[((size_t)t * p.H + head) * p.VD + col], beta = p.b.beta[(size_t)t * p.H + head], qk = p.b.qk[(size_t)t * p.KH + kvh];
    if (p.v.seg_pos[seg] == 0) s0 = s1 = f32x4 {0.f, 0.f, 0.f, 0.f};
    float a = 0.0f, b = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        s0[r] *= g0[r], s1[r] *= g1[r];
        a = fmaf(k0[r], s0[r], a), b = fmaf(q0[r], s0[r], b);
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) a = fmaf(k1[r], s1[r], a), b = fmaf(q1[r], s1[r], b);
    a = group_sum<L>(a), b = group_sum<L>(b);
    const float u = beta * (v - a);
#pragma unroll
    for (int r = 0; r < 4; ++r) s0[r] = fmaf(k0[r], u, s0[r]), s1[r] = fmaf(k1[r], u, s1[r]);
    *(f32x4 *)(state + 4 * li) = s0, *(f32x4 *)(state + 4 * (L + li)) = s1;
    if (li == 0) p.b.o[((size_t)t * p.H + head) * p.VD + col] = fmaf(qk, u, b);
}

struct OutParams {
    const float *o, *gates, *norm;
    const void *row_gate; // the gate in the rows of the input product (pitch ld), through a silu; or null
    int ld;
    void *out; // rows of pitch out_ld
    int out_ld;
    int H, VD, vdim, gcols, T;
    float eps, mul;
};

// per-head RMS norm times the gate; one wave a (token, head)
template <bool BF16>
__global__ __launch_bounds__(256) void delta_output_kernel(OutParams p) {
    const int lane = threadIdx.x & 63;
    const size_t idx = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (idx >= (size_t)p.T * p.H) return;
    const int t = (int)(idx / p.H), head = (int)(idx % p.H);
    const float *o = p.o + idx * p.VD;
    const float *gate = p.gates + (size_t)t * 2 * p.gcols + p.gcols + head * p.VD;
    float sq = 0.0f;
    for (int c = lane * 2; c < p.VD; c += 128) {
        const float2 x = *(const float2 *)(o + c);
        sq = fmaf(x.x, x.x, fmaf(x.y, x.y, sq));
    }
    const float r = 1.0f / sqrtf(wave_total(sq) / (float)p.vdim + p.eps);
    const float f = r * p.mul;
    for (int c = lane * 2; c < p.VD; c += 128) {
        const float2 x = *(const float2 *)(o + c), w = *(const float2 *)(p.norm + c);
        float2 z;
        if (p.row_gate) {
            z = load2<BF16>(p.row_gate, (size_t)t * p.ld + head * p.VD + c);
            z.x = silu_of<BF16>(z.x), z.y = silu_of<BF16>(z.y);
        } else {
            z = *(const float2 *)(gate + c);
            z.x = sigmoid_of<BF16>(z.x), z.y = sigmoid_of<BF16>(z.y);
        }
        store2<BF16>(p.out, (size_t)t * p.out_ld + head * p.VD + c, make_float2(x.x * f * w.x * z.x, x.y * f * w.y * z.y));
    }
}

// A step of one token a sequence, from the input product's rows to the output product's: convolutions, norms, decays, the state's step and the gated norm of a
// key head's heads in one workgroup, where the state of a head fits its registers (16 floats a thread).  The channels of a token are spread over the threads
// (q | k | v | decays, 256 each) and meet in LDS; the state is requested in front of that work, so that it arrives behind it.  A key head's workgroup alone
// touches its convolution inputs, which it shifts in place.  Every wave adds up the norms and q . k of the head by itself, over the same lanes as the
// separate launches do, so that the results are theirs bit for bit (by way of LDS, where 16 waves at once queue for it, 1 to 8 % of a step more).
// Bound by latency (a chain of two loads, two barriers, a store): a step of 16 heads of 128 x 128 in three launches / in one,
// six layers of it, BF16: 1 sequence 146 / 118 us, 4 174 / 138, 16 221 / 173, 64 458 / 403; 64 x 64 140 / 108 .. 243 / 247, 64 x 256 166 / 129 .. 483 / 420.
template <bool BF16, int L, bool ONE>
__global__ __launch_bounds__(1024) void delta_decode_kernel(PrepParams p, OutParams out) {
    constexpr int DT = BF16 ? XFTHIP_BF16 : XFTHIP_F32, KD = 8 * L, COLS = 1024 / L;
    __shared__ __align__(16) float qs[KD], ks[KD], gs[KD], vs[256], os[256];
    const int seg = blockIdx.x, kvh = blockIdx.y, each = p.H / p.KH, tid = threadIdx.x, lane = tid & 63;
    const int t = p.v.seg_off[seg], row = p.v.seg_row[seg], start = p.v.seg_pos[seg];
    const int li = tid % L, col0 = tid / L, role = tid >> 8, c = tid & 255, taps = p.taps;
    const size_t hist = (size_t)row * (taps - 1) * p.channels, in_row = (size_t)t * p.ld;
    f32x4 q0, q1, k0, k1;
    float qk = 0.0f;
    for (int r = 0; r < each; ++r) {
        const int head = kvh * each + r;
        const int ch = (role == 2 ? 2 * p.KH : role * p.KH + kvh) * KD + (role == 2 ? head * p.VD : 0) + c;
        const bool conv = role == 2 ? c < p.VD : role < 2 && r == 0 && c < KD, gate = role == 3 && !ONE && c < KD;
        float x[3] = {0.0f, 0.0f, 0.0f}, w[4] = {0.0f, 0.0f, 0.0f, 0.0f}, in = 0.0f, dt = 0.0f;
        if (conv) { // (x, w: the last three of at most four taps)
            in = ldb<BF16>(p.b.in, in_row + ch);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (j >= 4 - taps) w[j] = p.conv[(size_t)ch * taps + j - (4 - taps)];
#pragma unroll
            for (int j = 0; j < 3; ++j)
                if (j >= 4 - taps && start - 3 + j >= 0) x[j] = ldb<BF16>(p.b.conv_state, hist + (size_t)(j - (4 - taps)) * p.channels + ch);
        }
        if (gate) in = p.b.gates[(size_t)t * 2 * p.gcols + head * KD + c], dt = p.dt_bias[head * KD + c];
        if (ONE && role == 3) in = ldb<BF16>(p.b.in, in_row + p.decay_col + head), dt = p.dt_bias[head];
        const float decay = p.decay[head], beta = sigmoid_of<BF16>(ldb<BF16>(p.b.in, in_row + p.beta_col + head));
        float z = 0.0f, ow = 0.0f;
        if (tid < p.VD) {
            z = out.row_gate ? ldb<BF16>(out.row_gate, (size_t)t * out.ld + head * p.VD + tid) : out.gates[(size_t)t * 2 * out.gcols + out.gcols + head * p.VD + tid];
            ow = out.norm[tid];
        }
        float *state = p.b.state + ((size_t)row * p.H + head) * p.VD * KD + 4 * li;
        f32x4 s[2][2];
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            const int col = col0 + n * COLS;
            s[n][0] = s[n][1] = f32x4 {0.f, 0.f, 0.f, 0.f};
            if (col < p.VD && start > 0) s[n][0] = *(const f32x4 *)(state + (size_t)col * KD), s[n][1] = *(const f32x4 *)(state + (size_t)col * KD + 4 * L);
        }
        if (conv) {
            float a = 0.0f;
#pragma unroll
            for (int j = 0; j < 3; ++j) a = fmaf(w[j], x[j], a);
            a = silu_of<BF16>(fmaf(w[3], in, a));
#pragma unroll
            for (int j = 0; j < 3; ++j)
                if (j >= 4 - taps) store_from_f32(p.b.conv_state, DT, hist + (size_t)(j - (4 - taps)) * p.channels + ch, j < 2 ? x[j + 1] : in);
            (role == 0 ? qs : role == 1 ? ks : vs)[c] = a;
        }
        if (gate || (ONE && role == 3 && c == 0)) gs[c] = exp_of<BF16>(-decay * softplus_of<BF16>(in + dt));
        __syncthreads();
        if (r == 0) {
            float sq = 0.0f, sk = 0.0f;
#pragma unroll
            for (int i = 2 * lane; i < KD; i += 128) {
                const float2 x = *(const float2 *)(qs + i), y = *(const float2 *)(ks + i);
                sq = fmaf(x.x, x.x, fmaf(x.y, x.y, sq)), sk = fmaf(y.x, y.x, fmaf(y.y, y.y, sk)), qk = fmaf(x.x, y.x, fmaf(x.y, y.y, qk));
            }
            sq = 1.0f / sqrtf(wave_total_dpp(sq) + 1e-6f) * p.qscale, sk = 1.0f / sqrtf(wave_total_dpp(sk) + 1e-6f);
            qk = wave_total_dpp(qk) * sq * sk;
            q0 = *(const f32x4 *)(qs + 4 * li), q1 = *(const f32x4 *)(qs + 4 * (L + li)), k0 = *(const f32x4 *)(ks + 4 * li), k1 = *(const f32x4 *)(ks + 4 * (L + li));
#pragma unroll
            for (int i = 0; i < 4; ++i) q0[i] *= sq, q1[i] *= sq, k0[i] *= sk, k1[i] *= sk;
        }
        f32x4 g0, g1;
        if constexpr (ONE) {
            const float fade = gs[0];
            g0 = g1 = f32x4 {fade, fade, fade, fade};
        } else g0 = *(const f32x4 *)(gs + 4 * li), g1 = *(const f32x4 *)(gs + 4 * (L + li));
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            const int col = col0 + n * COLS;
            if (col >= p.VD) continue; // (whole groups of L lanes)
            f32x4 s0 = s[n][0] * g0, s1 = s[n][1] * g1;
            float a = 0.0f, b = 0.0f;
#pragma unroll
            for (int i = 0; i < 4; ++i) a = fmaf(k0[i], s0[i], a), b = fmaf(q0[i], s0[i], b);
#pragma unroll
            for (int i = 0; i < 4; ++i) a = fmaf(k1[i], s1[i], a), b = fmaf(q1[i], s1[i], b);
            a = group_sum<L>(a), b = group_sum<L>(b);
            const float u = beta * (vs[col] - a);
#pragma unroll
            for (int i = 0; i < 4; ++i) s0[i] = fmaf(k0[i], u, s0[i]), s1[i] = fmaf(k1[i], u, s1[i]);
            *(f32x4 *)(state + (size_t)col * KD) = s0, *(f32x4 *)(state + (size_t)col * KD + 4 * L) = s1;
            if (li == 0) os[col] = fmaf(qk, u, b);
        }
        __syncthreads();
        if (tid < (p.VD + 63) / 64 * 64) { // (whole waves; each adds up all of the head by itself)
            float sq = 0.0f;
            for (int i = 2 * lane; i < p.VD; i += 128) {
                const float2 x = *(const float2 *)(os + i);
                sq = fmaf(x.x, x.x, fmaf(x.y, x.y, sq));
            }
            const float f = 1.0f / sqrtf(wave_total_dpp(sq) / (float)out.vdim + out.eps) * out.mul;
            z = out.row_gate ? silu_of<BF16>(z) : sigmoid_of<BF16>(z);
            if (tid < p.VD) store_from_f32(out.out, DT, (size_t)t * out.out_ld + head * p.VD + tid, os[tid] * f * ow * z);
        }
    }
}

PrepParams prep_params(int act, const PlanLayer &L, const StepView &v, const DeltaBuffers &b) {
    PrepParams p;
    p.v = v, p.b = b, p.below = INT_MAX;
    p.b.in = (char *)b.in + (size_t)L.in_col * (act == XFTHIP_BF16 ? 2 : 4);
    p.conv = L.conv, p.decay = L.decay, p.dt_bias = L.dt_bias;
    p.H = L.s.heads, p.KH = L.s.kv_heads, p.KD = L.KD, p.VD = L.VD, p.taps = L.s.taps;
    p.ld = L.in_ld, p.channels = L.channels(), p.beta_col = L.channels(), p.decay_col = L.head_decay() ? p.beta_col + L.beta_cols() : -1, p.gcols = L.gcols;
    p.qscale = 1.0f / sqrtf((float)L.s.dim);
    return p;
}

// tiles of 16 columns of the states of so many segments: four waves each and more
long chunk_tiles(const PlanLayer &L, size_t segments) { return (long)segments * L.s.heads * (L.VD / 16); }

// launches over some of the segments: f(how many, which)
template <typename F>
void over_segments(const std::vector<int> &segments, F f) {
    for (size_t at = 0; at < segments.size(); at += kChunkSegs) {
        ChunkSegs s = {};
        const size_t n = std::min<size_t>(kChunkSegs, segments.size() - at);
        std::copy_n(segments.begin() + at, n, s.seg);
        f((unsigned)n, s);
    }
}

// row_in: the input product's rows, if the gate is in them
OutParams out_params(int act, const PlanLayer &L, int T, const float *o, const float *gates, const void *row_in, void *out, float eps) {
    const int esz = act == XFTHIP_BF16 ? 2 : 4;
    OutParams p = {o, gates, L.out_norm, row_in ? (const char *)row_in + (size_t)L.out_gate_col() * esz : nullptr, L.in_ld, (char *)out + (size_t)L.out_col * esz, L.out_ld};
    p.H = L.s.heads, p.VD = L.VD, p.vdim = L.s.vdim, p.gcols = L.gcols, p.T = T, p.eps = eps, p.mul = L.mix_scale;
    return p;
}

int launch_output(int act, const OutParams &p, int T, hipStream_t st) {
    const unsigned blocks = (unsigned)(((size_t)T * p.H + 3) / 4);
    if (act == XFTHIP_BF16) hipLaunchKernelGGL(delta_output_kernel<true>, dim3(blocks), dim3(256), 0, st, p);
    else hipLaunchKernelGGL(delta_output_kernel<false>, dim3(blocks), dim3(256), 0, st, p);
    XFT_CHECK_HIP(hipGetLastError());
    return 0;
}

} // namespace

// Which segments kChunk tokens at a time?
// Where all tiles of the step leave most of the device idle: all, from a longest of a whole chunk on (16 heads of 128 x 128, one prompt of 16 / 32 tokens 26 / 31 us token by token, so 21 / 22).
// Else, with hardly any short ones, all from two chunks on (16 prompts of 16 / 24 / 32 tokens 39 / 46 / 51 and 37 / 46 / 46), with one decay a head, which saves the walk a third of its reads, from
// eight (32 heads, 16 prompts of 32 / 64 / 400 tokens 65 / 104 / 603 and 66 / 107 / 526).
// Else each by its own length, since a single token costs as much as a whole chunk there; two launches more, which segments of less than four (eight) chunks do not pay for.  All token by token / all in
// chunks / so, us: one prompt of 64 / 128 / 500 tokens beside 50 decoding sequences 62 / 119 / 63, 83 / 168 / 58 and 196 / 467 / 84, beside 200 163 / 440 / 131, 222 / 624 / 137 and 249 / 1701 / 156; 4 of 300
// beside 20 170 / 125 / 91; with one decay a head, 32 heads, 128 tokens beside 50 101 / 243 / 84.
DeltaSplit delta_split(const PlanLayer &L, const StepView &v, const int *lens, bool chunks) {
    DeltaSplit s;
    s.rest = v.longest;
    if (!chunks || v.longest < kChunk || L.KD < 64 || L.KD > 256 || L.s.taps < 2 || L.s.taps > 4) return s;
    const long full = 4L * device_cu_count();
    const bool idle = chunk_tiles(L, v.B) < full;
    int from = idle ? kChunk : L.head_decay() ? 8 * kChunk : 2 * kChunk;
    const bool all = idle || chunk_tiles(L, std::count_if(lens, lens + v.B, [&](int n) { return n < from; })) < full / 2;
    if (!all) from = L.head_decay() ? 8 * kChunk : 4 * kChunk;
    if (v.longest < from) return s;
    s.rest = 0, s.longest = v.longest, s.below = from;
    for (int i = 0; i < v.B; ++i) {
        if (all || lens[i] >= from) s.by_chunks.push_back(i);
        else s.rest = std::max(s.rest, lens[i]);
    }
    return s;
}

int delta_prepare(int act, const PlanLayer &L, const StepView &v, const DeltaSplit &split, const DeltaBuffers &b, hipStream_t st) {
    PrepParams p = prep_params(act, L, v, b);
    const dim3 grid(v.T, (p.H + 3) / 4);
    const int width = p.KD > p.VD ? p.KD : p.VD;
    const bool tiled = p.taps >= 2 && p.taps <= 4 && width <= 256;
    if (!split.by_chunks.empty()) {
        auto launch = [&](auto bf16, auto f32) {
            over_segments(split.by_chunks, [&](unsigned n, const ChunkSegs &segs) {
                const dim3 chunks((split.longest + kChunk - 1) / kChunk, p.H, n);
                if (act == XFTHIP_BF16) hipLaunchKernelGGL(bf16, chunks, dim3(256), 0, st, p, segs);
                else hipLaunchKernelGGL(f32, chunks, dim3(256), 0, st, p, segs);
            });
        };
        switch (L.KD + (L.head_decay() ? 1 : 0)) {
            case 64: launch(delta_chunk_kernel<64, false, true>, delta_chunk_kernel<64, false, false>); break;
            case 65: launch(delta_chunk_kernel<64, true, true>, delta_chunk_kernel<64, true, false>); break;
            case 128: launch(delta_chunk_kernel<128, false, true>, delta_chunk_kernel<128, false, false>); break;
            case 129: launch(delta_chunk_kernel<128, true, true>, delta_chunk_kernel<128, true, false>); break;
            case 256: launch(delta_chunk_kernel<256, false, true>, delta_chunk_kernel<256, false, false>); break;
            default: launch(delta_chunk_kernel<256, true, true>, delta_chunk_kernel<256, true, false>); break;
        }
        XFT_CHECK_HIP(hipGetLastError());
        p.below = split.below;
        // (several workgroups read the inputs of a key head: nobody shifts those of a single token in place)
        if (!split.rest) return conv_tail(act, v, p.b.in, p.ld, p.channels, p.taps, b.conv_state, st, 1);
    }
    if (tiled) {
        const dim3 tiles((split.rest + kPrepTokens - 1) / kPrepTokens, (p.H + 3) / 4, v.B);
        const int key = (act == XFTHIP_BF16 ? 0 : 10) + p.taps + (width > 128 ? 100 : 0);
        switch (key) {
            case 2: hipLaunchKernelGGL((delta_prepare_tiled_kernel<true, 2, 1>), tiles, dim3(256), 0, st, p); break;
            case 3: hipLaunchKernelGGL((delta_prepare_tiled_kernel<true, 3, 1>), tiles, dim3(256), 0, st, p); break;
            case 4: hipLaunchKernelGGL((delta_prepare_tiled_kernel<true, 4, 1>), tiles, dim3(256), 0, st, p); break;
            case 12: hipLaunchKernelGGL((delta_prepare_tiled_kernel<false, 2, 1>), tiles, dim3(256), 0, st, p); break;
            case 13: hipLaunchKernelGGL((delta_prepare_tiled_kernel<false, 3, 1>), tiles, dim3(256), 0, st, p); break;
            case 14: hipLaunchKernelGGL((delta_prepare_tiled_kernel<false, 4, 1>), tiles, dim3(256), 0, st, p); break;
            case 102: hipLaunchKernelGGL((delta_prepare_tiled_kernel<true, 2, 2>), tiles, dim3(256), 0, st, p); break;
            case 103: hipLaunchKernelGGL((delta_prepare_tiled_kernel<true, 3, 2>), tiles, dim3(256), 0, st, p); break;
            case 104: hipLaunchKernelGGL((delta_prepare_tiled_kernel<true, 4, 2>), tiles, dim3(256), 0, st, p); break;
            case 112: hipLaunchKernelGGL((delta_prepare_tiled_kernel<false, 2, 2>), tiles, dim3(256), 0, st, p); break;
            case 113: hipLaunchKernelGGL((delta_prepare_tiled_kernel<false, 3, 2>), tiles, dim3(256), 0, st, p); break;
            default: hipLaunchKernelGGL((delta_prepare_tiled_kernel<false, 4, 2>), tiles, dim3(256), 0, st, p); break;
        }
    }
    if (!tiled) {
        if (act == XFTHIP_BF16) hipLaunchKernelGGL(delta_prepare_kernel<true>, grid, dim3(256), 0, st, p);
        else hipLaunchKernelGGL(delta_prepare_kernel<false>, grid, dim3(256), 0, st, p);
    }
    XFT_CHECK_HIP(hipGetLastError());
    return conv_tail(act, v, p.b.in, p.ld, p.channels, p.taps, b.conv_state, st);
}

int conv_tail(int act, const StepView &v, const void *in, int ld, int channels, int taps, void *conv_state, hipStream_t st, int least) {
    if (v.longest <= 1 || taps <= 1) return 0;
    const TailParams p = {v, in, ld, channels, taps, conv_state, least};
    const dim3 grid((channels + 255) / 256, v.B);
    if (act == XFTHIP_BF16) hipLaunchKernelGGL(conv_tail_kernel<true>, grid, dim3(256), 0, st, p);
    else hipLaunchKernelGGL(conv_tail_kernel<false>, grid, dim3(256), 0, st, p);
    XFT_CHECK_HIP(hipGetLastError());
    return 0;
}

size_t delta_chunk_floats(const PlanLayer &L, int tokens, int segments) {
    if (L.KD < 64 || L.KD > 256 || L.s.taps < 2 || L.s.taps > 4 || tokens < kChunk) return 0;
    return (size_t)(tokens / kChunk + std::min(segments, tokens)) * L.s.heads * chunk_floats(L.KD);
}

int delta_scan(const PlanLayer &L, const StepView &v, const DeltaSplit &split, const DeltaBuffers &b, hipStream_t st) {
    ScanParams p;
    p.v = v, p.b = b, p.H = L.s.heads, p.KH = L.s.kv_heads, p.VD = L.VD, p.below = INT_MAX;
    const int lanes = L.KD / 8;
    const bool one = L.head_decay();
    if (!split.by_chunks.empty()) {
        // Two tiles a wave where a CU has several workgroups of one in turn: 16 heads of 128 x 128, one / two, 4 prompts of 1000 to 1500 tokens 255 / 262 us, 6 of 200 to 1000 239 / 270, 8 of
        // 800 342 / 308, 16 of 400 351 / 314; 64 x 64, whose workgroups are of half the waves, 16 of 400 134 / 140; 8 of 256 x 256, 8 of 800 484 / 439
        const bool two = chunk_tiles(L, split.by_chunks.size()) >= (L.KD == 64 ? 8L : 4L) * device_cu_count(); // (value widths are whole 32s)
        auto scan = [&](auto one_tile, auto two_tiles, int waves) {
            over_segments(split.by_chunks, [&](unsigned n, const ChunkSegs &segs) {
                hipLaunchKernelGGL(two ? two_tiles : one_tile, dim3(n, p.H, L.VD / 16 / (two ? 2 : 1)), dim3(64 * waves + 64), 0, st, p, segs);
            });
        };
        switch (L.KD) {
            case 64: scan(delta_chunk_scan_kernel<64, 2, 1>, delta_chunk_scan_kernel<64, 2, 2>, 2); break;
            case 128: scan(delta_chunk_scan_kernel<128, 4, 1>, delta_chunk_scan_kernel<128, 4, 2>, 4); break;
            default: scan(delta_chunk_scan_kernel<256, 4, 1>, delta_chunk_scan_kernel<256, 4, 2>, 4); break;
        }
        XFT_CHECK_HIP(hipGetLastError());
        if (!split.rest) return 0;
        p.below = split.below;
    }
    // Two columns a group of lanes where one would make four waves a SIMD or more: below, the columns' chains are better hidden by each other's waves.  16
    // heads of 128 x 128, one column / two: 4 prompts of 1500 tokens 350 / 407 us, 6 of 1000 308 / 368, 8 of 800 308 / 272, 24 of 500 650 / 510.
    const bool two = split.rest > 1 && lanes >= 8 && L.VD % (512 / lanes) == 0 && (long)v.B * p.H * L.VD * lanes >= (long)device_cu_count() * 1024;
    const int cols = (two ? 512 : 256) / lanes;
    const dim3 grid(v.B, p.H, (L.VD + cols - 1) / cols);
    auto launch = [&](auto several, auto single) {
        if (one) hipLaunchKernelGGL(single, grid, dim3(256), 0, st, p);
        else hipLaunchKernelGGL(several, grid, dim3(256), 0, st, p);
    };
    const int key = (split.rest == 1 ? 0 : two ? 2000 : 1000) + L.KD;
    switch (key) {
        case 32: launch(delta_step_kernel<4, false>, delta_step_kernel<4, true>); break;
        case 64: launch(delta_step_kernel<8, false>, delta_step_kernel<8, true>); break;
        case 128: launch(delta_step_kernel<16, false>, delta_step_kernel<16, true>); break;
        case 256: launch(delta_step_kernel<32, false>, delta_step_kernel<32, true>); break;
        case 1032: launch(delta_scan_kernel<4, 2, 1, false>, delta_scan_kernel<4, 2, 1, true>); break;
        case 1064: launch(delta_scan_kernel<8, 2, 1, false>, delta_scan_kernel<8, 2, 1, true>); break;
        case 1128: launch(delta_scan_kernel<16, 2, 1, false>, delta_scan_kernel<16, 2, 1, true>); break;
        case 1256: launch(delta_scan_kernel<32, 2, 1, false>, delta_scan_kernel<32, 2, 1, true>); break;
        case 2064: launch(delta_scan_kernel<8, 2, 2, false>, delta_scan_kernel<8, 2, 2, true>); break;
        case 2128: launch(delta_scan_kernel<16, 2, 2, false>, delta_scan_kernel<16, 2, 2, true>); break;
        case 2256: launch(delta_scan_kernel<32, 2, 2, false>, delta_scan_kernel<32, 2, 2, true>); break;
        default: set_error("delta_scan: key dimension %d of a head is above 256", L.s.dim); return 2;
    }
    XFT_CHECK_HIP(hipGetLastError());
    return 0;
}

int delta_output(int act, const PlanLayer &L, const StepView &v, const DeltaBuffers &b, float eps, hipStream_t st) {
    if (L.silu_gate()) return gated_head_norm(act, L, v.T, b.o, b.in, b.out, eps, st);
    return launch_output(act, out_params(act, L, v.T, b.o, b.gates, nullptr, b.out, eps), v.T, st);
}

// The state of a head in the registers of one workgroup.  A second head of a key head follows the first in its workgroup: of the 29 and 40 us that six layers
// of 16 x 128 x 128 save at 1 and 4 sequences 14 and 16 are left with 8 key heads (38 of 49 at 16, 72 of 60 at 64); a third would take what is left.
// Smaller states only as long as a CU, which holds two workgroups, gets few after each other: a workgroup of 1024 threads takes as long for a small state as for a
// large one.  Three launches / one, six layers of 16 heads, 32 / 64 / 128 / 256 sequences: 32 x 32 184 / 168 us, 203 / 218, 224 / 308, 255 / 474; 64 x 64 220 / 190, 243 /
// 248, 280 / 336, 431 / 620; 64 x 128 242 / 211, 306 / 286, 437 / 482, 621 / 755; 128 x 96 254 / 220, 369 / 350, 510 / 505, 783 / 795; 128 x 128 272 / 245, 457 / 405, 594 / 559,
// 935 / 900.  (8192 values in three rounds 1 to 7 % slower, 4096 in two 2 %.)
bool delta_decodes_at_once(const PlanLayer &L, const StepView &v) {
    const int size = L.KD * L.VD, most = 2 * device_cu_count(), rounds = (v.B * L.s.kv_heads + most - 1) / most;
    return v.longest == 1 && L.s.taps >= 2 && L.s.taps <= 4 && L.KD <= 256 && L.VD <= 256 && size <= 16 * 1024 && L.s.heads <= 2 * L.s.kv_heads
            && (size == 16 * 1024 || rounds <= (size >= 12 * 1024 ? 4 : size >= 8 * 1024 ? 2 : 1));
}

int delta_decode(int act, const PlanLayer &L, const StepView &v, const DeltaBuffers &b, float eps, hipStream_t st) {
    const PrepParams p = prep_params(act, L, v, b);
    const OutParams out = out_params(act, L, v.T, nullptr, b.gates, L.silu_gate() ? b.in : nullptr, b.out, eps);
    const dim3 grid(v.B, p.KH);
    const bool one = L.head_decay();
    auto launch = [&](auto several, auto single) {
        if (one) hipLaunchKernelGGL(single, grid, dim3(1024), 0, st, p, out);
        else hipLaunchKernelGGL(several, grid, dim3(1024), 0, st, p, out);
    };
    switch ((act == XFTHIP_BF16 ? 0 : 1000) + L.KD) {
        case 32: launch(delta_decode_kernel<true, 4, false>, delta_decode_kernel<true, 4, true>); break;
        case 64: launch(delta_decode_kernel<true, 8, false>, delta_decode_kernel<true, 8, true>); break;
        case 128: launch(delta_decode_kernel<true, 16, false>, delta_decode_kernel<true, 16, true>); break;
        case 256: launch(delta_decode_kernel<true, 32, false>, delta_decode_kernel<true, 32, true>); break;
        case 1032: launch(delta_decode_kernel<false, 4, false>, delta_decode_kernel<false, 4, true>); break;
        case 1064: launch(delta_decode_kernel<false, 8, false>, delta_decode_kernel<false, 8, true>); break;
        case 1128: launch(delta_decode_kernel<false, 16, false>, delta_decode_kernel<false, 16, true>); break;
        case 1256: launch(delta_decode_kernel<false, 32, false>, delta_decode_kernel<false, 32, true>); break;
        default: set_error("delta_decode: key dimension %d of a head is above 256", L.s.dim); return 2;
    }
    XFT_CHECK_HIP(hipGetLastError());
    return 0;
}

int gated_head_norm(int act, const PlanLayer &L, int T, const float *o, const void *in, void *out, float eps, hipStream_t st) {
    return launch_output(act, out_params(act, L, T, o, nullptr, in, out, eps), T, st);
}

} // namespace xfthip
