// Causal GQA attention over the KV cache: decode (one new token), prefill and chunked
// prefill in one kernel.  Replaces the reference's crossAttnByHead / crossAttnShardedHead /
// selfScaledDpAttention (src/kernels/attention_kernels.h) and their small_gemm* helpers.
//
// Work decomposition.  The "columns" of a workgroup are up to 16 (query token, query head)
// pairs that share one KV head (for decode: the G heads of a GQA group).  Keys and values
// stream from HBM exactly once per column group:
//   S^T[token][col] = K[token][:] . Q[col][:]        MFMA 16x16x32 f16, A = K tile (16 tokens
//                                                     x 32 dims, one 128-bit load per lane)
//   O^T[dim][col]  += V^T[dim][token] . P^T[token][col]   A = V tile from the token-innermost
//                                                     value layout, B = probabilities straight
//                                                     from the score registers
// Scores, running max / sum and the output accumulate in fp32 (online softmax).  The KV
// sequence is split over gridDim.x workgroups and over the 4 waves of each; partial
// (max, sum, O) triples are merged in LDS and, across workgroups, by whichever workgroup of
// the column group finishes last (ticket counter, no spinning), the same statistic merge crossAttnShardedHead does (attention_kernels.h:931-983).
// INT8 caches are widened to fp16 in registers (exact); the per-token key scale multiplies
// the score column, the value scale multiplies the probability (gemm_kernel_ext.cpp:471-500,
// gemm_kernel_ext2.cpp:75-91).
#include <atomic>
#include <mutex>


#include "attention_dev.h"
#include "attention_prefill.h"

namespace xfthip {

// launch bounds: three workgroups a CU.  The next block's keys are requested as soon as this block's scores are
// scaled and its values once this block's P.V products are issued, into the registers those have just left; at 128
// registers (four workgroups a CU) the compiler spills to keep that order and everything is slower, at 168 it fits
// (146 FP16, 168 INT8).  Against four workgroups a CU that request each block only when they need it: INT8 cache,
// batch 64 x 16384 tokens 594 -> 388 us (5.7 TB/s), 16 x 4096 42 -> 30 us; FP16 725 -> 713 us (6.0 TB/s), 16 x 4096
// 61 -> 44 us, 64 x 1024 58 -> 48 us.
// With at most one block a wave (short contexts at small batches) nothing can be requested ahead: that form keeps
// the plain order, the shorter program (few workgroups then: the same launch bounds do no harm).
template <bool INT8, bool PIPE>
__global__ __launch_bounds__(256, 3) void attn_kernel(AttnParams p) {
    __shared__ AttnLds<4> lds;
    attn_unit<INT8, 4, PIPE>(p, blockIdx.x, blockIdx.y % p.kv.H, blockIdx.y / p.kv.H, blockIdx.z, lds, [] { __syncthreads(); });
}

// Short contexts: one workgroup of 8 waves, nothing split.  The hand-over between the workgroups of a split (publish, ticket, read back) is three round
// trips to memory, which two blocks more a wave do not cost.
template <bool INT8>
__global__ __launch_bounds__(512) void attn_short_kernel(AttnParams p) {
    __shared__ AttnLds<8> lds;
    attn_unit<INT8, 8, false>(p, 0, blockIdx.x % p.kv.H, blockIdx.x / p.kv.H, blockIdx.y, lds, [] { __syncthreads(); });
}

constexpr int kTicketParts = 8, kMaxParts = 32;
// merges the parts of a launch of attn_kernel that took no tickets: grid (columns of a group, groups), at most 128 parts
__global__ __launch_bounds__(128) void attn_merge_kernel(AttnParams p) {
    __shared__ float s_pm[128], s_f[128];
    attn_merge_unit(p, blockIdx.y, blockIdx.x, s_pm, s_f);
}

// 32 columns a wave, K / V blocks shared through LDS (attention_prefill.h); two workgroups a CU
template <bool INT8, bool FINE>
__global__ __launch_bounds__(256, 2) void attn_prefill32_kernel(AttnParams p, int ncg, int npairs, PrefillBands bands) {
    __shared__ __attribute__((aligned(16))) unsigned char lds[INT8 ? kRingLdsInt8 : kRingLds];
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    int first, width;
    prefill_band(bands, slot / ncg, first, width);
    const int at = slot - first * ncg, pair = (first + at % width) * 8 + xcd;
    if (pair >= npairs) return;
    attn_prefill_ring_unit<INT8, FINE>(p, pair % p.kv.H, ncg - 1 - at / width, pair / p.kv.H, lds);
}

// Split-KV merge workspace: `slots` partial-result slots of kSlotFloats floats and one ticket per
// column group.  Plain xfthip_attention calls take one per stream from the library's per-stream scratch
// (allocated on a stream's first call); a model owns its own.
int attention_workspace_create(AttnWorkspace *w, int slots) {
    w->ws = nullptr, w->tickets = nullptr, w->slots = 0;
    XFT_CHECK_HIP(hipMalloc((void **)&w->ws, (size_t)slots * kSlotFloats * sizeof(float)));
    XFT_CHECK_HIP(hipMalloc((void **)&w->tickets, (size_t)slots * sizeof(unsigned int)));
    XFT_CHECK_HIP(hipMemset(w->tickets, 0, (size_t)slots * sizeof(unsigned int)));
    XFT_CHECK_HIP(hipDeviceSynchronize());
    w->slots = slots;
    return 0;
}

void attention_workspace_destroy(AttnWorkspace *w) {
    if (w->ws) (void)hipFree(w->ws);
    if (w->tickets) (void)hipFree(w->tickets);
    w->ws = nullptr, w->tickets = nullptr, w->slots = 0;
}

// the workspace of plain calls on `stream`
int attention_stream_workspace(hipStream_t stream, AttnWorkspace *w) {
    void *parts = nullptr, *tickets = nullptr;
    if (int rc = stream_scratch(kScratchAttnParts, stream, (size_t)kWsSlots * kSlotFloats * sizeof(float), false, &parts)) return rc;
    if (int rc = stream_scratch(kScratchAttnTickets, stream, (size_t)kWsSlots * sizeof(unsigned int), true, &tickets)) return rc;
    w->ws = (float *)parts, w->tickets = (unsigned int *)tickets, w->slots = kWsSlots;
    return 0;
}

// ---- statically allocated workspace of xfthip_attention_static ---------------------------------
// Device memory that exists from the moment the code object is loaded: callers that must not
// allocate (stream capture, serving loops that forbid hipMalloc) get the split-KV partials and the
// tickets from here.  Each device holds its own copy at its own address; in host code the array's
// name is only a handle for hipGetSymbolAddress, never a pointer to pass to a kernel.
constexpr int kStaticSlots = 1024;
constexpr size_t kStaticTicketOffset = (size_t)kStaticSlots * kSlotFloats * sizeof(float);
static __device__ __align__(256) unsigned char scratch[kStaticTicketOffset + (size_t)kStaticSlots * sizeof(unsigned int)];

constexpr int kMaxDevices = 64;
static std::atomic<void *> g_scratch_ptr[kMaxDevices] = {}; // written once under g_scratch_mu, read without it
static std::mutex g_scratch_mu;

// Resolves (once per device, with that device current) the device address of `scratch` and clears
// the tickets.  Allocates nothing.  Called by xfthip_init and by the entry point's first call on a device.
int attention_static_scratch_init() {
    int dev = -1;
    XFT_CHECK_HIP(hipGetDevice(&dev));
    XFT_REQUIRE(dev >= 0 && dev < kMaxDevices, "attention_static_scratch_init: device index %d out of range", dev);
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_ptr[dev].load(std::memory_order_acquire) != nullptr) return 0;
    void *ptr = nullptr;
    XFT_CHECK_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    XFT_REQUIRE(ptr != nullptr, "attention_static_scratch_init: no device address for the static scratch");
    XFT_CHECK_HIP(hipMemset((unsigned char *)ptr + kStaticTicketOffset, 0, (size_t)kStaticSlots * sizeof(unsigned int)));
    XFT_CHECK_HIP(hipDeviceSynchronize());
    g_scratch_ptr[dev].store(ptr, std::memory_order_release);
    return 0;
}

} // namespace xfthip

using namespace xfthip;

// len_hint: upper bound of the visible sequence length when the positions live in device memory
// (0 = unknown, the cache length is assumed); it only steers the split count.
// wsp: the workspace to merge splits through (nullptr = the library's shared one, allocated on first
// use).  strict: fail instead of lowering the split count when the workspace is too small.
int xfthip::attention_launch(xfthip_kvcache_t c, const void *q, int qStride, void *out, int oStride, int out_dtype, int B, int S,
        int qHeads, float scale, int past, const int *past_dev, int len_hint, hipStream_t stream, const AttnWorkspace *wsp,
        bool strict) {
    XFT_REQUIRE(c && q && out, "xfthip_attention: null argument");
    XFT_REQUIRE(B > 0 && B <= c->kv.B, "xfthip_attention: batch %d exceeds cache batch %d", B, c->kv.B);
    XFT_REQUIRE(S > 0 && qHeads > 0 && qHeads % c->kv.H == 0, "xfthip_attention: bad S=%d or qHeads=%d (kvHeads=%d)", S, qHeads,
            c->kv.H);
    XFT_REQUIRE(c->kv.D == 128, "xfthip_attention: head size %d unsupported", c->kv.D);
    XFT_REQUIRE(out_dtype == XFTHIP_BF16 || out_dtype == XFTHIP_F32, "xfthip_attention: out_dtype must be bf16 or f32");
    XFT_REQUIRE(qStride >= qHeads * 128 && (qStride % 8) == 0 && ((uintptr_t)q & 15) == 0,
            "xfthip_attention: q must be 16-byte aligned with qStride >= qHeads*128 and %% 8 == 0");
    XFT_REQUIRE(oStride >= qHeads * 128, "xfthip_attention: oStride too small");
    XFT_REQUIRE(past_dev != nullptr || (past >= 0 && past + S <= c->maxSeq),
            "xfthip_attention: past %d + S %d exceeds the cache length %d", past, S, c->maxSeq);
    AttnParams p = {};
    p.kv = c->kv;
    p.q = (const uint16_t *)q;
    p.qStride = qStride;
    p.out = out;
    p.oStride = oStride;
    p.out_dtype = out_dtype;
    p.B = B;
    p.S = S;
    p.G = qHeads / c->kv.H;
    p.scale = scale;
    p.past = past;
    p.past_dev = past_dev;
    p.CG = (S * p.G + 15) / 16;
    // many columns per KV head (prefill, long chunks)
    {
        const int form = attention_prefill_form(c->kv.int8, p.G, (long)B * c->kv.H, S, past);
        if (form) {
            p.nsplit = 1;
            const int ncg = (S * p.G + 127) / 128, npairs = B * c->kv.H;
            const PrefillBands bands = prefill_bands((npairs + 7) / 8);
            dim3 grid(8 * ((npairs + 7) / 8) * ncg);
            const bool fine = form == 2;
            if (c->kv.int8 && fine) hipLaunchKernelGGL((attn_prefill32_kernel<true, true>), grid, dim3(256), 0, stream, p, ncg, npairs, bands);
            else if (c->kv.int8) hipLaunchKernelGGL((attn_prefill32_kernel<true, false>), grid, dim3(256), 0, stream, p, ncg, npairs, bands);
            else if (fine) hipLaunchKernelGGL((attn_prefill32_kernel<false, true>), grid, dim3(256), 0, stream, p, ncg, npairs, bands);
            else hipLaunchKernelGGL((attn_prefill32_kernel<false, false>), grid, dim3(256), 0, stream, p, ncg, npairs, bands);
            XFT_CHECK_HIP(hipGetLastError());
            return 0;
        }
    }
    // split the KV sequence so that the launch has about one workgroup a CU (attention_split_count); the longest
    // visible sequence is bounded by the cache length when the real one lives in device memory
    const int len = past_dev ? ((len_hint > 0 && len_hint < c->maxSeq) ? len_hint : c->maxSeq) : past + S;
    const int wgs = B * c->kv.H * p.CG;
    int nsplit = attention_split_count(len, wgs);
    AttnWorkspace of_stream;
    if (nsplit > 1) {
        if (wsp == nullptr) {
            if (int rc = attention_stream_workspace(stream, &of_stream)) return rc;
            wsp = &of_stream;
        }
        if ((size_t)wgs * nsplit > (size_t)wsp->slots) {
            XFT_REQUIRE(!strict,
                    "xfthip_attention_static: %d column groups x %d sequence splits need %zu partial-result slots, the static "
                    "scratch holds %d; use xfthip_attention for this shape",
                    wgs, nsplit, (size_t)wgs * nsplit, wsp->slots);
            while (nsplit > 1 && (size_t)wgs * nsplit > (size_t)wsp->slots) --nsplit;
        }
    }
    // (Behind the workspace all the same: a stream's first call takes it, so that a longer one can be captured later.)
    if (attention_short(c->kv.int8, p.G, len, nsplit)) {
        p.nsplit = 1;
        const dim3 grid(c->kv.H * p.CG, B);
        if (c->kv.int8) hipLaunchKernelGGL(attn_short_kernel<true>, grid, dim3(512), 0, stream, p);
        else hipLaunchKernelGGL(attn_short_kernel<false>, grid, dim3(512), 0, stream, p);
        XFT_CHECK_HIP(hipGetLastError());
        return 0;
    }
    p.nsplit = nsplit;
    p.ws = wsp ? wsp->ws : nullptr;
    // up to kTicketParts parts the last workgroup of a column group merges them; beyond, a second launch does (8 KV
    // heads, 2048 tokens, 16 parts: 11.7 us merged by the last workgroup, 10.2 by the launch; 4096 tokens 13.7 / 12.7)
    const bool merge_launch = nsplit > kTicketParts;
    p.tickets = (wsp && !merge_launch) ? wsp->tickets : nullptr;
    dim3 grid(nsplit, c->kv.H * p.CG, B);
    // more than one 32-token block a wave somewhere: the form that requests blocks ahead
    const bool pipe = (len + 31) / 32 > 4 * nsplit;
    if (c->kv.int8) {
        if (pipe) hipLaunchKernelGGL((attn_kernel<true, true>), grid, dim3(256), 0, stream, p);
        else hipLaunchKernelGGL((attn_kernel<true, false>), grid, dim3(256), 0, stream, p);
    } else {
        if (pipe) hipLaunchKernelGGL((attn_kernel<false, true>), grid, dim3(256), 0, stream, p);
        else hipLaunchKernelGGL((attn_kernel<false, false>), grid, dim3(256), 0, stream, p);
    }
    if (merge_launch) {
        const int cols = S * p.G < 16 ? S * p.G : 16;
        hipLaunchKernelGGL(attn_merge_kernel, dim3(cols, wgs), dim3(128), 0, stream, p);
    }
    XFT_CHECK_HIP(hipGetLastError());
    return 0;
}

bool xfthip::attention_short(bool int8, int G, int len, int nsplit) {
    // Up to 320 tokens, and 384 of a cache half as large or with several query heads a KV head, 8 waves of one workgroup are faster than the parts of a
    // split and their merge; beyond, a CU's own path to the L2 takes longer than the merge.  FP16, one sequence, 32 KV heads, 176 / 256 / 320 / 512 tokens:
    // split 7.4 / 7.6 / 7.7 / 8.0 us, so 6.1 / 6.8 / 7.4 / 9.2; 8 KV heads of 32: 8.5 / 8.9 / 9.0 / 9.2 and 6.5 / 7.1 / 7.8 / 9.6; INT8, 32 KV heads: 7.3
    // / 7.5 / 7.5 / 7.8 and 6.1 / 6.3 / 7.0 / 8.7, at 384 7.5 and 7.1.  Batches and portions (FP16 and INT8, 1 to 31 sequences, 1 to 8 new tokens, 8 to 64 query heads, 130 to
    // 400 tokens, 1356 shapes) took 0.43 to 1.0 times as long, 0.71 in the mean: the more column groups, the more a split's hand-over cost (16 sequences of 130 tokens, 4 new, 32 / 8
    // heads, INT8 17.7 and 7.6 us).
    return nsplit > 1 && len <= (int8 || G > 1 ? 384 : 320);
}

int xfthip::attention_split_count(int len, int units) {
    // Measured over batch 1 .. 64, 8 and 32 KV heads, 512 .. 16384 tokens, both cache kinds: a launch is fastest with
    // about one workgroup a CU.  With at least that many (batch, KV head, column group) units nothing is split, and the
    // partials, tickets and merge fall away with it (64 sequences x 8 KV heads x 512 tokens: 35 -> 27 us FP16, 26 ->
    // 17 us INT8, against two parts); below, the sequence is cut into CUs / units parts, twice that where this gives
    // at most 4 parts and the sequence has 2048 tokens or more (16 x 8 KV heads x 4096 tokens INT8: 37.5 us with 2
    // parts, 32.8 with 4), every wave keeping at least one 32-token block, 32 parts at most (batch 1, 8 KV heads,
    // 16384 tokens: 23.0 us with 16 parts, 20.2 with 32, 23.0 with 64; INT8 21.6 / 16.2 / 16.9).
    const int nblk = (len + 31) / 32;
    const int cus = device_cu_count();
    if (units >= cus) return 1;
    int nsplit = cus / units;
    if (nsplit <= 4 && nblk >= 64) nsplit *= 2;
    const int cap = (nblk + 3) / 4;
    if (nsplit > cap) nsplit = cap;
    if (nsplit > kMaxParts) nsplit = kMaxParts;
    if (nsplit < 1) nsplit = 1;
    while (nsplit > 1 && (size_t)units * nsplit > (size_t)kWsSlots) --nsplit;
    return nsplit;
}

extern "C" int xfthip_attention(xfthip_kvcache_t c, const void *q, int qStride, void *out, int oStride, int out_dtype,
        int B, int S, int qHeads, float scale, int past, const int *past_dev, xfthip_stream_t stream) {
    return attention_launch(c, q, qStride, out, oStride, out_dtype, B, S, qHeads, scale, past, past_dev, 0, (hipStream_t)stream,
            nullptr, false);
}

extern "C" int xfthip_attention_static(xfthip_kvcache_t c, const void *q, int qStride, void *out, int oStride, int out_dtype,
        int B, int S, int qHeads, float scale, int past, const int *past_dev, xfthip_stream_t stream) {
    int dev = -1;
    XFT_CHECK_HIP(hipGetDevice(&dev));
    XFT_REQUIRE(dev >= 0 && dev < kMaxDevices, "xfthip_attention_static: device index %d out of range", dev);
    if (g_scratch_ptr[dev].load(std::memory_order_acquire) == nullptr)
        if (int rc = attention_static_scratch_init()) return rc;
    unsigned char *base = (unsigned char *)g_scratch_ptr[dev].load(std::memory_order_acquire);
    AttnWorkspace w;
    w.ws = (float *)base;
    w.tickets = (unsigned int *)(base + kStaticTicketOffset);
    w.slots = kStaticSlots;
    return attention_launch(c, q, qStride, out, oStride, out_dtype, B, S, qHeads, scale, past, past_dev, 0, (hipStream_t)stream, &w,
            true);
}
