// moe_batched.hip — the MoE layer for T tokens at once on gfx950 (the
// reference's run_moe_batched, src/glm_layer_runner.cuh:818-928, used by
// prefill): an expert's weights are read once per pass of up to 64 of its tokens
// instead of once per token.
//
//   bnorm    RMSNorm per token -> norm (f32) and, for a bf16 shared expert, norm3
//            (its three bf16 pieces)
//   broute   router logits, kTB tokens per work-group; norm and logits use the
//            arithmetic of the decode and routing kernels, so a token's ids
//            equal the ones wl_run_moe selects for it
//   btopk    sigmoid + bias, top-k, weights (one work-group per token), and the
//            token's row of norm quantised in place (q6.h)
//   bcount   per expert: its entries (token*K + slot) in ascending order
//            (wave ballots, deterministic) and their count
//   bscatter per expert: its compact range (prefix of the counts), ent/pos
//            (calls of few entries: both inside bup, group_entries)
//   bup      gate/up + SwiGLU: shared expert (unit = token pass x 64 or 128 rows),
//            routed experts (unit = expert pass x 4 x 64 rows) -> midf, compact
//            rows; a routed pass's activation DMAs read its tokens' quantised rows
//            in place, through tables of tokens in LDS
//   bquant   the rows of midf quantised -> mid6
//   bdown    down: shared expert (unit = token pass x 128 or 256 rows), routed
//            experts (unit = expert pass x 512 rows) -> expout
//   bcomb    out[t] = (resid[t] +) sum_k w[t][k] e_k[t] (slot order) + shared[t]
//
// The routed GEMMs run each activation as 6-bit pieces against the MXFP4 weights as
// they are on the scaled matrix instruction (q6.h), the bf16 shared expert's as three
// bf16 pieces (x = p0 + p1 + p2 to f32 precision) through v_mfma_f32_16x16x32_bf16.
// bup and bdown are persistent (one work-group per CU) and share one step pipeline
// (batched_gemm.h): activations arrive in LDS by DMA, weights two steps ahead in
// registers. A dense layer of many positions has kernels of its own (batched_dense.h).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "dev_common.h"
#include "internal.h"
#include "q6.h"

namespace wl {

#define WL_MEM __device__ __forceinline__  // member functions

constexpr uint32_t kTB = 8;          // tokens per routing work-group

constexpr uint32_t kGW = 8;         // waves of a GEMM work-group
constexpr uint32_t kGT = 64 * kGW;  // its threads

// split3 of any value: one past bf16's largest starts with that (rounded to
// infinity it would leave -infinity to the other pieces, and a NaN), an infinity
// is its first piece alone.
WL_DEV void split3_any(float x, uint32_t& h, uint32_t& m, uint32_t& l) {
    const uint32_t u = __float_as_uint(x);
    h = f2bf(x);
    if ((h & 0x7FFFu) == 0x7F80u) h = u >> 16;
    const float r1 = (u & 0x7FFFFFFFu) == 0x7F800000u ? 0.f : x - bf2f(h);
    m = f2bf(r1);
    l = f2bf(r1 - bf2f(m));
}
// The three bf16 pieces of 4 consecutive values at p, p + stride, p + 2 stride
// (ANY: of values that may leave bf16's range).
template <bool ANY = false>
WL_DEV void store_pieces4(uint16_t* p, uint32_t stride, const float (&x)[4]) {
    uint32_t h[4], md[4], l[4], mx = 0u;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        split3(x[q], h[q], md[q], l[q]);
        mx = max(mx, __float_as_uint(x[q]) & 0x7FFFFFFFu);
    }
    if (ANY && mx >= 0x7F7F8000u) {  // (rounds to infinity)
#pragma unroll
        for (int q = 0; q < 4; q++) split3_any(x[q], h[q], md[q], l[q]);
    }
    auto pack = [](const uint32_t (&x)[4]) {
        return (uint64_t)(x[0] | (x[1] << 16)) | ((uint64_t)(x[2] | (x[3] << 16)) << 32);
    };
    gst((uint64_t*)p, pack(h));
    gst((uint64_t*)(p + stride), pack(md));
    gst((uint64_t*)(p + 2u * stride), pack(l));
}

// ---- routing ------------------------------------------------------------------
// RMSNorm of token t = blockIdx.x (norm_rinv / norm_value: the decode kernel's
// arithmetic) into b.norm, and its three bf16 pieces into b.norm3 (for a bf16
// shared expert).
__global__ void __launch_bounds__(kThreads) bnorm_kernel(const DecodeArgs* __restrict__ pa, const BatchArgs b) {
    const DecodeArgs& a = *pa;
    const uint32_t H = a.H, tid = threadIdx.x, t = blockIdx.x;
    __shared__ float red[kWaves * 64];
    const rsrc_t hid_rs = make_rsrc(b.hidden + (size_t)t * H, H * 4u);
    const rsrc_t ln_rs = make_rsrc(a.ln_w ? (const void*)a.ln_w : (const void*)b.hidden, H * 2u);
    float4 hv[kHV];
    uint2 lv[kHV];
#pragma unroll
    for (int i = 0; i < kHV; i++) {
        const uint32_t j = tid + kThreads * i;
        hv[i] = __builtin_bit_cast(float4, bld16(hid_rs, 16u * j, 0u));
        lv[i] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(ln_rs, (int)(8u * j), 0, 0));
    }
    if (t == 0u && tid < 2u) gst(b.more + tid, 0u);  // (the kernels after this one set them)
    const float rinv = norm_rinv(hv, red, H, a.eps);
#pragma unroll
    for (int i = 0; i < kHV; i++) {
        const uint32_t j = tid + kThreads * i;
        if (j < H / 4) {
            const float xs[4] = {hv[i].x, hv[i].y, hv[i].z, hv[i].w};
            const uint32_t ls[4] = {lv[i].x & 0xFFFFu, lv[i].x >> 16, lv[i].y & 0xFFFFu, lv[i].y >> 16};
            float4 o;
            o.x = norm_value(xs[0], rinv, a.ln_w != nullptr, ls[0]);
            o.y = norm_value(xs[1], rinv, a.ln_w != nullptr, ls[1]);
            o.z = norm_value(xs[2], rinv, a.ln_w != nullptr, ls[2]);
            o.w = norm_value(xs[3], rinv, a.ln_w != nullptr, ls[3]);
            *(__attribute__((address_space(1))) u32x4*)(b.norm + (size_t)t * b.ldn + 4 * j) = __builtin_bit_cast(u32x4, o);
            const float os[4] = {o.x, o.y, o.z, o.w};
            if (!(b.flags & kBatchShared4)) store_pieces4(b.norm3 + (size_t)t * 3u * H + 4 * j, H, os);
        }
    }
}

// Wave sums of NV values per lane at once (NV a power of two <= 64), each
// summed over the 64 lanes by the same tree as router_partial_x's butterfly
// (x += shfl_xor(x, o), o = 32, 16, ..., 1): at each of the first log2(NV)
// levels a lane keeps half of its values and adds its partner's copy of them
// (the two operands the butterfly adds in this lane at this level), the
// levels after that are the butterfly itself. Afterwards lane l holds, in
// x[0], the sum of value l >> (6 - log2 NV) — bit for bit the butterfly's.
// (Levels are template parameters: every index into x is a constant, so x
// stays in registers without indexed moves.)
template <uint32_t N, uint32_t n, uint32_t o>  // values [0, 2n) -> [0, n) at offset o
WL_DEV void wave_levels(float (&x)[N]) {
    if constexpr (n >= 1u) {
        const bool up = (threadIdx.x & o) != 0u;
#pragma unroll
        for (uint32_t j = 0; j < n; j++) {
            const float keep = up ? x[j + n] : x[j];
            const float send = up ? x[j] : x[j + n];
            x[j] = keep + __shfl_xor(send, (int)o, 64);
        }
        wave_levels<N, n / 2u, o / 2u>(x);
    } else if constexpr (o >= 1u) {
        x[0] += __shfl_xor(x[0], (int)o, 64);
        wave_levels<N, 0u, o / 2u>(x);
    }
}
template <uint32_t NV>
WL_DEV void multi_wave_sum(float (&x)[NV]) {
    static_assert(NV >= 1u && NV <= 64u && (NV & (NV - 1u)) == 0u, "NV: a power of two <= 64");
    wave_levels<NV, NV / 2u, 32u>(x);
}

// Router logits of kTB tokens: each thread keeps its router_chain_x share of
// every token's normalised input in registers; the rows stream through, kRR
// at a time (rows r = x + gridDim.x (kRR i + q), q < kRR; the next group
// prefetched). The kRR x kTB wave sums of a group are taken together
// (multi_wave_sum), then summed over the waves in order from 0 — the
// arithmetic of router_partial and router_publish, so each logit equals the
// one the decode and routing kernels compute for the token.
constexpr uint32_t kRR = 4;  // router rows per group
__global__ void __launch_bounds__(kThreads) broute_kernel(const DecodeArgs* __restrict__ pa, const BatchArgs b) {
    const DecodeArgs& a = *pa;
    const uint32_t H = a.H, E = a.E, tid = threadIdx.x, lane = tid & 63u, v = uni(tid >> 6);
    constexpr uint32_t NV = kRR * kTB;  // value q * kTB + tt: row q, token tt
    constexpr uint32_t SH = 6u - __builtin_ctz(NV);
    constexpr uint32_t kFL = 64;  // groups whose logits are buffered in LDS
    __shared__ float red[kWaves * 64];
    __shared__ float lgb[kFL * NV];
    const uint32_t t0 = blockIdx.y * kTB, nch = H / 8, gx = gridDim.x;
    float4 xr[kTB][kRCH][2];  // xn[8c .. 8c+8) of chunks c = tid + 512 m, per token
#pragma unroll
    for (uint32_t tt = 0; tt < kTB; tt++) {
        const bool live = t0 + tt < b.T;
        const rsrc_t nrs = make_rsrc(b.norm + (size_t)min(t0 + tt, b.T - 1u) * b.ldn, live ? H * 4u : 0u);
#pragma unroll
        for (int m = 0; m < kRCH; m++) {
            const uint32_t c = tid + kThreads * m;
            xr[tt][m][0] = __builtin_bit_cast(float4, bld16(nrs, 32u * c, 0u));
            xr[tt][m][1] = __builtin_bit_cast(float4, bld16(nrs, 32u * c + 16u, 0u));
        }
    }
    const rsrc_t rt_rs = make_rsrc(a.router_w, E * H * 2u);
    auto row_of = [&](uint32_t i, uint32_t q) { return blockIdx.x + gx * (kRR * i + q); };
    u32x4 rn[kRR][kRCH];
#pragma unroll
    for (uint32_t q = 0; q < kRR; q++)
#pragma unroll
        for (int m = 0; m < kRCH; m++)
            rn[q][m] = bld16(rt_rs, 16u * min(tid + kThreads * m, nch - 1u), min(row_of(0u, q), E - 1u) * H * 2u);
    for (uint32_t i = 0; row_of(i, 0u) < E; i++) {
        u32x4 rw[kRR][kRCH];
#pragma unroll
        for (uint32_t q = 0; q < kRR; q++)
#pragma unroll
            for (int m = 0; m < kRCH; m++) {
                rw[q][m] = rn[q][m];
                rn[q][m] = bld16(rt_rs, 16u * min(tid + kThreads * m, nch - 1u), min(row_of(i + 1u, q), E - 1u) * H * 2u);
            }
        // router_chain_x for every (row, token) value, its chunks in the same
        // order (m, then the 8 columns), with one branch per chunk instead of
        // one per value, so the NV independent chains interleave
        float x[NV];
#pragma unroll
        for (uint32_t j = 0; j < NV; j++) x[j] = 0.f;
#pragma unroll
        for (int m = 0; m < kRCH; m++) {
            if (tid + kThreads * m < nch) {
#pragma unroll
                for (uint32_t q = 0; q < kRR; q++) {
                    const u32x4 r = rw[q][m];
                    const float wv[8] = {bf2f(r.x & 0xFFFFu), bf2f(r.x >> 16), bf2f(r.y & 0xFFFFu), bf2f(r.y >> 16),
                                         bf2f(r.z & 0xFFFFu), bf2f(r.z >> 16), bf2f(r.w & 0xFFFFu), bf2f(r.w >> 16)};
#pragma unroll
                    for (uint32_t tt = 0; tt < kTB; tt++) {
                        const float4 x0 = xr[tt][m][0], x1 = xr[tt][m][1];
                        float pd = x[q * kTB + tt];
                        pd = fmaf(wv[0], x0.x, pd);
                        pd = fmaf(wv[1], x0.y, pd);
                        pd = fmaf(wv[2], x0.z, pd);
                        pd = fmaf(wv[3], x0.w, pd);
                        pd = fmaf(wv[4], x1.x, pd);
                        pd = fmaf(wv[5], x1.y, pd);
                        pd = fmaf(wv[6], x1.z, pd);
                        pd = fmaf(wv[7], x1.w, pd);
                        x[q * kTB + tt] = pd;
                    }
                }
            }
        }
        multi_wave_sum(x);
        if ((lane & ((1u << SH) - 1u)) == 0u) red[v * 64u + (lane >> SH)] = x[0];
        lds_barrier();
        if (tid < NV) {
            float sum = 0.f;  // the same order as router_publish
#pragma unroll
            for (int wv = 0; wv < kWaves; wv++) sum += red[wv * 64 + tid];
            lgb[(i % kFL) * NV + tid] = sum;
        }
        lds_barrier();
        // the logits go out kFL groups at a time: a store in the loop would be
        // waited for with the next group's rows (loads and stores share one
        // counter), i.e. every group would wait for a store's round trip
        if (i % kFL == kFL - 1u || row_of(i + 1u, 0u) >= E) {
            const uint32_t i0 = i - i % kFL, n = (i % kFL + 1u) * NV;
            for (uint32_t j = tid; j < n; j += kThreads) {
                const uint32_t q = (j % NV) / kTB, tt = j % kTB, r = row_of(i0 + j / NV, q);
                if (r < E && t0 + tt < b.T) gst(b.logits + (size_t)(t0 + tt) * E + r, lgb[j]);
            }
        }
    }
}

// The top-k of token t = blockIdx.x, and its normalised row, which the router
// was the last to read, quantised in place (q6.h).
__global__ void __launch_bounds__(kThreads) btopk_kernel(const DecodeArgs* __restrict__ pa, const BatchArgs b) {
    const DecodeArgs& a = *pa;
    const uint32_t H = a.H, E = a.E, K = a.K, t = blockIdx.x, tid = threadIdx.x;
    __shared__ __align__(16) float row[(8192 / 32) * 36];  // 4 floats between blocks of 32: other banks
    __shared__ uint32_t wide;
    __shared__ double part[2][kWaves];
    float* rowp = b.norm + (size_t)t * b.ldn;
    for (uint32_t j = tid; j < H / 4u; j += kThreads) *(u32x4*)(row + 36u * (j / 8u) + 4u * (j % 8u)) = gld16(rowp + 4u * j);
    if (tid == 0u) wide = 0u;
    extern __shared__ __align__(16) uint8_t lds[];
    float* tk_sc = (float*)lds;
    float* tk_ch = tk_sc + E;
    uint32_t* tk_idx = (uint32_t*)(tk_ch + E);
    float* tk_w = (float*)(tk_idx + 32);
    for (uint32_t e = tid; e < E; e += kThreads)
        topk_score(gld(b.logits + (size_t)t * E + e), gld(a.bias + e), e, tk_sc, tk_ch);
    lds_barrier();  // (every thread's reads of the row are done)
    f32x16 even, odd;
    auto quantise = [&](uint32_t i) {
        if (i >= H / 32u) return;
        q6_load(row + 36u * i, even, odd);
        const uint32_t mx = q6_max(even, odd);
        if (q6_wide(even, odd, mx)) wide = 1u;
        q6_store<false>((uint8_t*)rowp + (i / 4u) * kQRecord, i % 4u, even, odd, mx);
    };
    // up to 256 experts the argmax is wave 0's: the other waves quantise (at most
    // 256 blocks)
    if (E <= 256u) {
        if (tid < 64u) topk_argmax_wave(E, K, tk_sc, tk_ch, tk_idx, tk_w);
        else quantise(tid - 64u);
    } else {
        topk_rank(E, K, tk_sc, tk_ch, tk_idx, tk_w);
        quantise(tid);
    }
    lds_barrier();
    if (tid < K) {
        gst(b.idx + (size_t)t * K + tid, (int32_t)tk_idx[tid]);
        gst(b.wts + (size_t)t * K + tid, topk_weight(a, K, tk_w, tid));
    }
    bool more = false;
    if (wide != 0u) {
        QRange rg{0.0, 0.0};
        if (tid < H / 32u) {
            q6_load(row + 36u * tid, even, odd);
            rg = q6_range(even, odd);
        }
        const double big = wave_sum_f64(rg.big), rest = wave_sum_f64(rg.rest);
        if ((tid & 63u) == 0u) {
            part[0][tid >> 6] = big;
            part[1][tid >> 6] = rest;
        }
        lds_barrier();
        double sb = 0.0, sr = 0.0;
        for (uint32_t w = 0; w < kWaves; w++) {
            sb += part[0][w];
            sr += part[1][w];
        }
        more = q6_more(sb, sr);
    }
    if (tid == 0u) gst(b.more_up + t, more ? 1u : 0u);
    if (!more) return;
    if (tid == 0u) gst(b.more, 1u);
    if (tid < H / 32u) {
        q6_load(row + 36u * tid, even, odd);
        q6_store<true>((uint8_t*)rowp + q6_row_bytes(H) + (tid / 4u) * kQMore, tid % 4u, even, odd, q6_max(even, odd));
    }
}

// Entries of expert e in ascending (token, slot) order: one wave, 64 entries
// per step, positions from a ballot prefix; the ids of kCB steps are loaded
// at once (one memory round trip per kCB steps).
constexpr uint32_t kCB = 8;
__global__ void __launch_bounds__(64) bcount_kernel(const BatchArgs b, uint32_t K) {
    const uint32_t e = blockIdx.x, lane = threadIdx.x, n = b.T * K;
    const rsrc_t ids = make_rsrc(b.idx, n * 4u);  // past n: zeros, masked by i < n
    uint32_t base = 0;
    for (uint32_t i0 = 0; i0 < n; i0 += 64u * kCB) {
        uint32_t id[kCB];
#pragma unroll
        for (uint32_t j = 0; j < kCB; j++)
            id[j] = __builtin_amdgcn_raw_buffer_load_b32(ids, (int)(4u * (i0 + 64u * j + lane)), 0, 0);
#pragma unroll
        for (uint32_t j = 0; j < kCB; j++) {
            const uint32_t i = i0 + 64u * j + lane;
            const bool hit = i < n && id[j] == e;
            const uint64_t bal = __builtin_amdgcn_ballot_w64(hit);
            const uint32_t below =
                __builtin_amdgcn_mbcnt_hi((uint32_t)(bal >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)bal, 0u));
            if (hit) gst(b.lists + (size_t)e * b.T + base + below, i);
            base += (uint32_t)__builtin_popcountll(bal);
        }
    }
    if (lane == 0) gst(b.counts + e, base);
}

// The compact range of expert e (exclusive prefix of the counts) and its
// entries' compact indices.
__global__ void __launch_bounds__(256) bscatter_kernel(const BatchArgs b, uint32_t E) {
    const uint32_t e = blockIdx.x, tid = threadIdx.x;
    __shared__ uint32_t s_off;
    if (tid < 64) {
        uint32_t s = 0;
        for (uint32_t f = tid; f < e; f += 64) s += gld(b.counts + f);
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        if (tid == 0) {
            s_off = s;
            gst(b.offsets + e, s);
            if (e == E - 1) gst(b.offsets + E, s + gld(b.counts + e));
        }
    }
    __syncthreads();
    const uint32_t off = s_off, ne = gld(b.counts + e);
    for (uint32_t i = tid; i < ne; i += blockDim.x) {
        const uint32_t en = gld(b.lists + (size_t)e * b.T + i);
        gst(b.ent + off + i, en);
        gst(b.pos + en, off + i);
    }
}

// ---- pass table ----------------------------------------------------------------
// An expert's tokens are cut into MFMA row blocks of 16, and those are split
// evenly over passes of at most kWide blocks (100 tokens: 7 blocks, 4 + 3).
constexpr uint32_t kRB = 16;                       // tokens of a row block
constexpr uint32_t kWide = 4;                      // row blocks of the largest pass
struct PassSplit {
    uint32_t np, base, rem;  // passes; the first rem of them have base + 1 row blocks, the others base
    // the passes of nb row blocks and the first of them
    WL_MEM uint32_t count(uint32_t nb) const { return np == 0u ? 0u : base == nb ? np - rem : base + 1u == nb ? rem : 0u; }
    WL_MEM uint32_t first(uint32_t nb) const { return base == nb ? rem : 0u; }
    // a bit for each size of pass that there is
    WL_MEM uint32_t sizes() const { return np == 0u ? 0u : 1u << base | (rem ? 2u << base : 0u); }
};
// (single: into passes of one block)
WL_DEV PassSplit pass_split(uint32_t c, bool single) {
    const uint32_t m = cdiv(c, kRB), np = single ? m : cdiv(m, kWide);
    if (np <= 1u) return PassSplit{np, m, 0u};  // (most: no division)
    return PassSplit{np, m / np, m % np};
}
// The experts' counts and offsets, in LDS, and room for the pass table.
// E counts the MXFP4 shared pseudo-expert (index E - 1) when there is one:
// all T tokens, compact rows from T*K on.
struct ExpertTab {
    uint32_t *cnt, *off, *pp;
    // each wave's, of its experts: bits of the sizes of this launch's passes; all
    // passes of the call | more of them if single << 16
    uint32_t *sizes, *sums;
};
// Pass table of the passes of nb row blocks: pp the exclusive prefix of the
// experts' passes, pp[E] all of them (rewritten for each nb). Units are numbered
// densely over the passes that exist (unit u = pass j * parts + part), so the
// grid-stride loop visits live units only and the passes of one expert sit next
// to each other.
struct PassTab {
    const uint32_t *cnt, *off, *pp;
    uint32_t n, nb;  // passes; row blocks of each
    bool single;
};
WL_DEV PassTab load_pass_tab(const ExpertTab& et, uint32_t E, uint32_t nb, bool single) {
    const uint32_t tid = threadIdx.x;
    lds_barrier();  // the tables are written, the last pass table is no longer read
    if (tid < 64u) {
        const uint32_t per = cdiv(E, 64u), e0 = tid * per;
        uint32_t mine = 0;
        for (uint32_t i = 0; i < per; i++)
            if (e0 + i < E) mine += pass_split(et.cnt[e0 + i], single).count(nb);
        uint32_t inc = mine;
#pragma unroll
        for (uint32_t o = 1; o < 64u; o <<= 1) {
            const uint32_t t0 = __shfl_up(inc, o, 64);
            if (tid >= o) inc += t0;
        }
        uint32_t run = inc - mine;
        for (uint32_t i = 0; i < per; i++)
            if (e0 + i < E) {
                et.pp[e0 + i] = run;
                run += pass_split(et.cnt[e0 + i], single).count(nb);
            }
        if (tid == 63u) et.pp[E] = inc;
    }
    lds_barrier();
    return PassTab{et.cnt, et.off, et.pp, uni(et.pp[E]), nb, single};
}
// Routed unit r (< n_passes * parts) -> (pass j, part). Units go in blocks
// of 8 passes x parts, ordered so that unit r has j % 8 == r % 8 in full
// blocks: with a grid of a multiple of 8 (work-group b runs on XCD b % 8),
// the units of one pass run on one XCD and share its L2 copy of the pass's
// activations.
struct PassPart {
    uint32_t j, part;
};
WL_DEV PassPart pass_part(uint32_t r, uint32_t parts, uint32_t npass) {
    const uint32_t blk = r / (8u * parts), l = r % (8u * parts);
    const uint32_t np = min(8u, npass - 8u * blk);
    return PassPart{8u * blk + l % np, l / np};
}
// Pass j (< n): its expert (the largest e with pp[e] <= j, which has a pass
// since pp[e + 1] > j), the pass within the expert, its token count and its
// first compact entry.
struct Pass {
    uint32_t e, nt, c0;
};
// (Counted by ballots: the reads do not depend on each other, where a binary
// search is eight round trips in a row for 256 experts.)
WL_DEV uint32_t expert_of_pass(const uint32_t* pp, uint32_t E, uint32_t j) {
    const uint32_t lane = threadIdx.x & 63u;
    uint32_t n = 0;
#pragma unroll 4
    for (uint32_t e0 = 0; e0 < E; e0 += 64u)
        n += (uint32_t)__builtin_popcountll(__builtin_amdgcn_ballot_w64(e0 + lane < E && pp[min(e0 + lane, E)] <= j));
    return n - 1u;
}
WL_DEV Pass pass_at(const PassTab& pt, uint32_t E, uint32_t j) {
    const uint32_t e = expert_of_pass(pt.pp, E, j), c = uni(pt.cnt[e]);
    const PassSplit sp = pass_split(c, pt.single);
    const uint32_t p = sp.first(pt.nb) + j - uni(pt.pp[e]), r0 = kRB * (p * sp.base + min(p, sp.rem));
    return Pass{e, min(kRB * pt.nb, c - r0), uni(pt.off[e]) + r0};
}

// ---- token table -------------------------------------------------------------
// A routed pass's activations are its tokens' quantised rows of norm, read in place by
// the DMAs. Before a gate/up pipeline runs, its work-group writes the tokens
// of its units' passes into LDS, tt[W i + m] = the token of row m of its unit
// i (W: the pipeline's largest pass), in one round of global loads for the
// whole pipeline; a unit's bind then reads its lanes' tokens there. (A call whose
// entries bup groups itself has the tokens of all entries there instead.) (A
// prefetch into registers would cost a wait at every bind: the compiler does
// not know how many steps lie between a load and its use.) The host sizes
// the table (BatchArgs::tcap entries) for the most units a work-group can
// get (batched_tok_entries); past it, tokens read as 0 and E_TOKTAB is raised.
template <class Kn>
WL_DEV void fill_tokens(const Kn& k, uint16_t* tt, uint32_t W) {
    if (k.nu * W > k.b.tcap && threadIdx.x == 0u) raise_error(k.a.sync, SyncMap::make(), E_TOKTAB, 0u);
    // wave v takes units v, v + kGW, ...: unit() takes a uniform index (it
    // reads the pass table through readfirstlane), lane m the pass rows m, m + 64
    const uint32_t v = uni(threadIdx.x >> 6), lane = threadIdx.x & 63u;
    constexpr uint32_t R = 4, M = (kRB * kWide + 63u) / 64u;  // units per wave whose loads are in flight together
    for (uint32_t i0 = 0; i0 < k.nu; i0 += R * kGW) {
        uint32_t ent[R][M];
        bool has[R][M];
#pragma unroll
        for (uint32_t r = 0; r < R; r++) {
            const uint32_t i = i0 + v + kGW * r;
#pragma unroll
            for (uint32_t j = 0; j < M; j++) has[r][j] = false;
            if (i < k.nu) {
                const auto x = k.unit(i);
#pragma unroll
                for (uint32_t j = 0; j < M; j++) {
                    const uint32_t m = lane + 64u * j;
                    has[r][j] = x.live && x.e != k.a.E && m < x.nt;
                    if (has[r][j]) ent[r][j] = k.b.ent[x.row0 + m];
                }
            }
        }
#pragma unroll
        for (uint32_t r = 0; r < R; r++) {
            const uint32_t i = i0 + v + kGW * r;
#pragma unroll
            for (uint32_t j = 0; j < M; j++) {
                const uint32_t m = lane + 64u * j;
                if (i < k.nu && m < W && W * i + m < k.b.tcap) tt[W * i + m] = (uint16_t)(has[r][j] ? ent[r][j] / k.K : 0u);
            }
        }
    }
    lds_barrier();
}
// The token of row m (< nt) of this work-group's unit i.
WL_DEV uint32_t table_token(const uint16_t* tt, uint32_t cap, uint32_t W, uint32_t i, uint32_t m, uint32_t nt) {
    const uint32_t idx = W * i + min(m, nt - 1u);
    return idx < cap ? (uint32_t)tt[idx] : 0u;
}

// Tables every GEMM work-group loads into LDS: the pass table and the
// layer's expert block pointers.
// With an MXFP4 shared expert, entry E is its block (NativeShared4::blk = 0).
WL_DEV const uint8_t* const* load_slot_tab(const DecodeArgs& a, uint32_t E, bool sh4, const uint8_t** s) {
    for (uint32_t f = threadIdx.x; f < E + (sh4 ? 1u : 0u); f += kGT)
        s[f] = f < E ? gld(a.slot_tab + f) : a.sh_native;
    return s;  // visible after the barrier in load_pass_tab
}
// LDS of the tables for E experts and the MXFP4 shared pseudo-expert.
__host__ __device__ inline size_t gemm_tab_bytes(uint32_t E) { return 8u * (E + 1u) + 4u * (4u * (E + 1u) + 2u); }
// The gate/up kernel's token table follows them (16-byte aligned).
__host__ __device__ inline size_t tok_table_offset(uint32_t E) { return (gemm_tab_bytes(E) + 15u) & ~(size_t)15u; }
// The dynamic LDS of the kernel (every extern __shared__ array starts there).
WL_DEV uint8_t* dyn_lds() {
    extern __shared__ __align__(16) uint8_t dyn_base[];
    return dyn_base;
}

WL_DEV void bld8(rsrc_t r, uint32_t voff, uint32_t soff, uint32_t (&s)[2]) {
    const uint2 v = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(r, (int)voff, (int)soff, 0));
    s[0] = v.x;
    s[1] = v.y;
}

#include "batched_gemm.h"
#include "batched_dense.h"

// The gate/up and down projections of every expert (persistent: the grid is
// what the chip holds at once, one work-group per CU).
__global__ void __launch_bounds__(kGT) bup_kernel(const DecodeArgs* __restrict__ pa, const BatchArgs b) {
    run_gemm<true>(pa, b);
}
__global__ void __launch_bounds__(kGT) bdown_kernel(const DecodeArgs* __restrict__ pa, const BatchArgs b) {
    run_gemm<false>(pa, b);
}

// The routed SwiGLU values (midf) as quantised rows (mid6, mid6x): a row per wave,
// one block of 32 values per lane, staged through LDS so that the loads are
// coalesced. Bound by the bytes (4096 tokens of inter 2048, 8 experts each: 590 MB in
// 112 us); where the experts come in groups, a group's rows and, with the first, the
// MXFP4 shared expert's alone (quant_rows).
struct QuantRows {
    uint32_t q0, qn, n;  // qn rows from q0, then the shared expert's (from T K on), n in all
};
__host__ __device__ inline QuantRows quant_rows(const BatchArgs& b, uint32_t K) {
    const bool part = (b.flags & kBatchSkipUnbound) != 0u;
    const uint32_t qn = part ? b.qn : b.T * K, sh = (b.flags & kBatchShared4) && !(b.flags & kBatchNoShared) ? b.T : 0u;
    return QuantRows{part ? b.q0 : 0u, qn, qn + sh};
}
__global__ void __launch_bounds__(256) bquant_kernel(const DecodeArgs* __restrict__ pa, const BatchArgs b) {
    const DecodeArgs& a = *pa;
    const uint32_t I = a.I, nb = I / 32u, lane = threadIdx.x & 63u, v = uni(threadIdx.x >> 6);
    const QuantRows qr = quant_rows(b, a.K);
    const uint32_t i0 = min(blockIdx.x * 4u + v, qr.n - 1u), row = i0 < qr.qn ? qr.q0 + i0 : b.T * a.K + i0 - qr.qn;
    const bool live = blockIdx.x * 4u + v < qr.n;
    __shared__ __align__(16) float xs[4][64 * 36];  // 32 values + 4: consecutive blocks in different banks
    const float* mid = b.midf + (size_t)row * b.ldm;
    f32x16 even, odd;
    bool wide = false;
    for (uint32_t b0 = 0; b0 < nb; b0 += 64u) {
#pragma unroll
        for (uint32_t i = 0; i < 8; i++) {
            const uint32_t c = lane + 64u * i;  // 16-byte chunk c % 8 of block c / 8
            *(u32x4*)(xs[v] + 36u * (c / 8u) + 4u * (c % 8u)) = gld16(mid + 32u * min(b0 + c / 8u, nb - 1u) + 4u * (c % 8u));
        }
        lds_barrier();
        const uint32_t k = b0 + lane;
        if (live && k < nb) {
            q6_load(xs[v] + 36u * lane, even, odd);
            const uint32_t mx = q6_max(even, odd);
            wide |= q6_wide(even, odd, mx);
            q6_store<false>(b.mid6 + (size_t)row * q6_row_bytes(I) + (k / 4u) * kQRecord, k % 4u, even, odd, mx);
        }
        lds_barrier();
    }
    bool more = false;
    if (__builtin_amdgcn_ballot_w64(wide) != 0u) {
        double big = 0.0, rest = 0.0;
        for (uint32_t k = lane; k < nb; k += 64u) {
            q6_load(mid + 32u * k, even, odd);
            const QRange rg = q6_range(even, odd);
            big += rg.big;
            rest += rg.rest;
        }
        more = q6_more(wave_sum_f64(big), wave_sum_f64(rest));
    }
    if (live && lane == 0u) {
        gst(b.more_dn + row, more ? 1u : 0u);
        if (more) gst(b.more + 1, 1u);
    }
    if (!live || !more) return;
    for (uint32_t k = lane; k < nb; k += 64u) {
        q6_load(mid + 32u * k, even, odd);
        q6_store<true>(b.mid6x + (size_t)row * q6_more_bytes(I) + (k / 4u) * kQMore, k % 4u, even, odd, q6_max(even, odd));
    }
}

// out[t] = (resid[t] +) sum_k w[t][k] e_k[t] in slot order + shared[t]
// (reference pass 3, src/glm_layer_runner.cuh:904-921).
// Thread: 4 consecutive rows (16-byte loads; H is a multiple of 128), each
// with the scalar sequence acc = fma(w_k, e_k, acc) over k, + shared, + resid.
__global__ void __launch_bounds__(256) bcomb_kernel(const BatchArgs b, uint32_t H, uint32_t K) {
    const uint32_t t = blockIdx.y;
    const uint32_t r = 4u * (blockIdx.x * blockDim.x + threadIdx.x);
    if (r >= H) return;
    float4 acc = {0.f, 0.f, 0.f, 0.f};
    for (uint32_t k = 0; k < K; k++) {
        const uint32_t c = gld(b.pos + (size_t)t * K + k);
        const float w = gld(b.wts + (size_t)t * K + k);
        const float4 x = *(const float4*)(b.expout + (size_t)c * b.ldm + r);
        acc.x = fmaf(w, x.x, acc.x);
        acc.y = fmaf(w, x.y, acc.y);
        acc.z = fmaf(w, x.z, acc.z);
        acc.w = fmaf(w, x.w, acc.w);
    }
    const float4 sh = (b.flags & kBatchShared4) ? *(const float4*)(b.expout + ((size_t)b.T * K + t) * b.ldm + r)
                                                : *(const float4*)(b.shout + (size_t)t * H + r);
    acc.x += sh.x;
    acc.y += sh.y;
    acc.z += sh.z;
    acc.w += sh.w;
    if (b.resid) {
        const float4 rs = *(const float4*)(b.resid + (size_t)t * H + r);
        acc.x = rs.x + acc.x;
        acc.y = rs.y + acc.y;
        acc.z = rs.z + acc.z;
        acc.w = rs.w + acc.w;
    }
    *(float4*)(b.out + (size_t)t * H + r) = acc;
}

// Token-table entries a work-group of the gate/up kernel can need for T
// tokens (an upper bound over every routing): R = T (K + 1) rows (K + 1 counts an
// MXFP4 shared expert's) make at most R / (16 (nb - 1) + 1) passes of nb row
// blocks, and at most one of one or two row blocks per expert, with a 32nd more where
// all passes have one block (run_gemm); a work-group gets at most cdiv(units, grid)
// of them.
static uint32_t batched_tok_entries(uint32_t T, uint32_t I, uint32_t E, uint32_t K, uint32_t grid) {
    auto cd = [](uint64_t a, uint64_t b) { return (a + b - 1u) / b; };
    const uint64_t R = (uint64_t)T * (K + 1u), NS = cd(I / kSlice, 4u);
    uint64_t most = 0;
    for (uint32_t nb = 1; nb <= kWide; nb++) {
        uint64_t n = R / (kRB * (nb - 1u) + 1u);
        if (nb <= 2u) n = std::min<uint64_t>(n, E + 1u + (E + 1u) / 32u + 1u);
        most = std::max(most, cd(n * NS, grid) * kRB * nb);
    }
    return (uint32_t)most;
}
static size_t bup_lds(uint32_t T, uint32_t I, uint32_t E, uint32_t K, uint32_t grid) {
    return tok_table_offset(E) + 2u * (size_t)batched_tok_entries(T, I, E, K, grid);
}
uint32_t batched_max_tokens(uint32_t I, uint32_t E, uint32_t K, uint32_t grid) {
    const size_t room = (size_t)decode_max_lds() - 3u * (size_t)kSlotB;
    uint32_t lo = 0, hi = 1u << 16;
    while (lo < hi) {
        const uint32_t mid = (lo + hi + 1u) / 2u;
        if (bup_lds(mid, I, E, K, grid) <= room) lo = mid;
        else hi = mid - 1u;
    }
    return lo;
}

uint32_t batched_max_experts() {
    // the GEMM kernels' LDS: the three activation slots and the expert tables
    const size_t lds = (size_t)decode_max_lds(), ring = 3u * (size_t)kSlotB;
    uint32_t e = 0;
    while (ring + gemm_tab_bytes(e + 16u) <= lds) e += 16u;
    return e;
}

int launch_batched(const DecodeArgs* d_args, const BatchArgs& b, uint32_t H, uint32_t I, uint32_t SI, uint32_t E,
                   uint32_t K, uint32_t n_cu, uint32_t phases, void* stream) {
    hipStream_t s = (hipStream_t)stream;
    hipError_t e;
    const size_t topk_lds = 4u * (2u * E + 64u);
    const size_t gemm_lds = gemm_tab_bytes(E);
    // the gate/up kernel's token table, sized for this call and a grid of
    // n_cu or more work-groups
    BatchArgs bt = b;
    bt.tcap = batched_tok_entries(b.T, I, E, K, n_cu);
    const size_t room = (size_t)decode_max_lds() - 3u * (size_t)kSlotB;
    bt.group = phases == kPhaseAll && !(b.flags & kBatchSkipUnbound) && b.T * K <= kGroupMax &&
               4u * E * group_words(b.T) <= kSlotB && tok_table_offset(E) + 2u * b.T * K <= room;
    const size_t up_lds = bt.group ? tok_table_offset(E) + 2u * b.T * K : bup_lds(b.T, I, E, K, n_cu);
    if (up_lds + 3u * (size_t)kSlotB > (size_t)decode_max_lds()) return (int)hipErrorInvalidValue;
    const void *up = (const void*)bup_kernel, *down = (const void*)bdown_kernel;
    const struct { const void* fn; size_t lds; } attrs[] = {
        {(const void*)btopk_kernel, topk_lds}, {up, up_lds}, {down, gemm_lds}};
    for (const auto& at : attrs)
        if ((e = hipFuncSetAttribute(at.fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)at.lds)) != hipSuccess)
            return (int)e;
    // The GEMM kernels walk their units with a grid stride, so their grid is
    // what the chip holds at once (the LDS ring allows one work-group per CU);
    // a larger grid would leave its second part waiting for the first.
    auto resident = [&](const void* fn, size_t lds) {
        int nb = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, fn, kGT, lds) != hipSuccess || nb < 1) nb = 1;
        return n_cu * (uint32_t)nb;
    };
    if (phases & kPhaseRoute) {
        hipLaunchKernelGGL(bnorm_kernel, dim3(b.T), dim3(kThreads), 0, s, d_args, b);
        // router: ~one work-group per CU; each token block's rows split over gx
        // work-groups (each norm row is read gx times, the router once per block)
        const uint32_t nblk = (b.T + kTB - 1) / kTB;
        const uint32_t gx = std::max(1u, std::min(n_cu / nblk, (E + kRR - 1) / kRR));
        hipLaunchKernelGGL(broute_kernel, dim3(gx, nblk), dim3(kThreads), 0, s, d_args, b);
        hipLaunchKernelGGL(btopk_kernel, dim3(b.T), dim3(kThreads), topk_lds, s, d_args, b);
        if (!bt.group) {
            hipLaunchKernelGGL(bcount_kernel, dim3(E), dim3(64), 0, s, b, K);
            hipLaunchKernelGGL(bscatter_kernel, dim3(E), dim3(256), 0, s, b, E);
        }
    }
    if (phases & kPhaseGemm) {
        const uint32_t gu = resident(up, up_lds), gd = resident(down, gemm_lds);
        const uint32_t rows = quant_rows(b, K).n;
        hipLaunchKernelGGL(bup_kernel, dim3(gu), dim3(kGT), up_lds, s, d_args, bt);
        if (rows) hipLaunchKernelGGL(bquant_kernel, dim3((rows + 3u) / 4u), dim3(256), 0, s, d_args, bt);
        hipLaunchKernelGGL(bdown_kernel, dim3(gd), dim3(kGT), gemm_lds, s, d_args, bt);
    }
    if (phases & kPhaseCombine)
        hipLaunchKernelGGL(bcomb_kernel, dim3((H + 1023) / 1024, b.T), dim3(256), 0, s, b, H, K);
    return (int)hipGetLastError();
}

uint64_t dense_token_bytes(uint32_t H, uint32_t DI) { return 6ull * H + 6ull * DI + 4ull * kDenseS * H; }
int launch_dense_batched(const DenseBatch& x, uint32_t n_cu, void* scratch, void* stream) {
    hipStream_t s = (hipStream_t)stream;
    auto cd = [](uint64_t a, uint64_t b) { return (a + b - 1u) / b; };
    // Passes and splits, in steps of a work-group (128 columns; 1.3 us with four
    // row blocks): its rounds of units times a unit's steps and about two for its
    // start, down also the partial rows written and read back at 5 TB/s. (200
    // positions of hidden 6144, inter 12288: five passes of 40 make 480 gate/up
    // units of three row blocks, two rounds of 256; four of 50 two rounds of four
    // row blocks.)
    uint32_t np = 0, S = 1;
    double best = 0.0;
    const uint64_t kup = cd(x.H, 128u), kdn = cd(x.DI, 128u);
    for (uint64_t p = cd(x.T, 64u); p <= cd(x.T, 16u); p++) {
        const double c = (double)(cd(cd(x.DI, 128u) * p, n_cu) * (kup + 2u)) * (1.0 + (double)cd(cd(x.T, p), kRB));
        if (np == 0u || c < best) {
            best = c;
            np = (uint32_t)p;
        }
    }
    for (uint32_t k = 1; k <= kDenseS; k++) {
        const double c = (double)(cd(cd(x.H, 256u) * np * k, n_cu) * (cd(kdn, k) + 2u)) + (double)k * x.T * x.H / 8.5e5;
        if (k == 1u || c < best) {
            best = c;
            S = k;
        }
    }
    DenseArgs d{x.hidden, x.resid, x.out, x.ln, x.gate, x.up, x.down, x.T, x.H, x.DI, np, S, x.eps, x.tap,
                (uint16_t*)scratch, nullptr, nullptr};
    d.mid3 = d.norm3 + 3ull * x.T * x.H;
    d.part = (float*)(d.mid3 + 3ull * x.T * x.DI);
    hipLaunchKernelGGL(dnorm_kernel, dim3(x.T), dim3(kThreads), 0, s, d);
    DenseArgs du = d;
    du.S = 1u;
    const uint32_t nb = (uint32_t)cd(cd(x.T, np), kRB);
#define WL_DENSE(NB)                                                              \
    case NB:                                                                      \
        hipLaunchKernelGGL((dgemm_kernel<true, NB>), dim3(n_cu), dim3(kGT), 0, s, du); \
        hipLaunchKernelGGL((dgemm_kernel<false, NB>), dim3(n_cu), dim3(kGT), 0, s, d); \
        break
    switch (nb) {
        WL_DENSE(1);
        WL_DENSE(2);
        WL_DENSE(3);
        WL_DENSE(4);
    }
#undef WL_DENSE
    hipLaunchKernelGGL(dsum_kernel, dim3((uint32_t)(((uint64_t)x.T * x.H / 4u + 255u) / 256u)), dim3(256), 0, s, d);
    return (int)hipGetLastError();
}

}  // namespace wl
