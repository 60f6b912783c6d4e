// The dense SwiGLU MLP over many positions (included by moe_batched.hip, inside
// namespace wl): bf16 weights row-major as the caller's files hold them, RMSNorm,
// gate/up, down and the residual in four launches. One position at a time (the
// attention library's dense MLP, 76 us each at hidden 6144, inter 12288) 200
// positions read the 453 MB of weights 200 times; here a pass of up to 64 positions
// reads them once.
//
// Arithmetic: three bf16 pieces of each activation (x = p0 + p1 + p2 to f32
// precision) through v_mfma_f32_16x16x32_bf16; every step's products sum in an
// accumulator that starts at zero and is added to the f32 sum, the roundings of
// which are kept (Knuth's two-sum) and added at the end: plain sums of 48 and 96
// steps had an error of 1.9e-7 against 64 bits, the one-position kernels 1.6e-7.
struct DenseArgs {
    const float *hidden, *resid;  // [T][H]; resid may be null
    float* out;                   // [T][H]; may be hidden or resid
    const uint16_t *ln, *gate, *up, *down;
    uint32_t T, H, DI, np, S;  // np: passes; S: K splits of down
    float eps;
    float* tap;       // the last position's normalised row (or null)
    uint16_t* norm3;  // [T][3][H] pieces
    uint16_t* mid3;   // [T][3][DI] pieces
    float* part;      // [S][T][H]
};
__global__ void __launch_bounds__(kThreads) dnorm_kernel(const DenseArgs d) {
    const uint32_t H = d.H, tid = threadIdx.x, t = blockIdx.x;
    __shared__ float red[kWaves * 64];
    const rsrc_t hid_rs = make_rsrc(d.hidden + (size_t)t * H, H * 4u);
    const rsrc_t ln_rs = make_rsrc(d.ln ? (const void*)d.ln : (const void*)d.hidden, H * 2u);
    float4 hv[kHV];
    uint2 lv[kHV];
#pragma unroll
    for (int i = 0; i < kHV; i++) {
        const uint32_t j = tid + kThreads * i;
        hv[i] = __builtin_bit_cast(float4, bld16(hid_rs, 16u * j, 0u));
        lv[i] = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(ln_rs, (int)(8u * j), 0, 0));
    }
    const float rinv = norm_rinv(hv, red, H, d.eps);
#pragma unroll
    for (int i = 0; i < kHV; i++) {
        const uint32_t j = tid + kThreads * i;
        if (j >= H / 4u) continue;
        const float os[4] = {norm_value(hv[i].x, rinv, d.ln != nullptr, lv[i].x & 0xFFFFu),
                             norm_value(hv[i].y, rinv, d.ln != nullptr, lv[i].x >> 16),
                             norm_value(hv[i].z, rinv, d.ln != nullptr, lv[i].y & 0xFFFFu),
                             norm_value(hv[i].w, rinv, d.ln != nullptr, lv[i].y >> 16)};
        store_pieces4(d.norm3 + (size_t)t * 3u * H + 4u * j, H, os);
        if (d.tap && t == d.T - 1u) gst((f32x4*)(d.tap + 4u * j), f32x4{os[0], os[1], os[2], os[3]});
    }
}

// Unit: a pass of the positions (split evenly over np passes, NB row
// blocks) x 8 waves x two tiles of 16 weight rows x one of the S splits of K. UP:
// tile 0 gate rows, tile 1 the same up rows, K = H, S = 1, SwiGLU values as pieces
// to mid3. Down: 32 output rows per wave, K = DI, f32 partial rows. A step is 128
// columns; a load takes 128 bytes, a cache line, of each of eight rows, and the
// lanes trade halves (rows_swap; 64 bytes of each of 16 rows: 1 % slower at 200
// positions, 4 % at 8 of hidden 2944, inter 6832). Columns past K and rows past the matrix are out of
// range: zeros on both sides. The slot is SharedK's. Bound by the LDS reads of
// the fragments and the matrix cores (each near 3100 cycles of a step with four
// row blocks) and, measured, the weight loads: 200 positions of hidden 6144, inter
// 12288 take 372 us (two thirds gate/up); one position at a time they took 15200.
template <bool UP, uint32_t NB>
struct DenseK {
    using AS = AStreamS;
    struct WB {
        u32x4 w[8];
    };
    static constexpr uint32_t kRows = UP ? 128u : 256u;  // matrix rows of a unit (UP: of both matrices)
    static constexpr uint32_t kLoads = 8, kRB2 = (NB + 1) / 2, kDmas = 3 * kRB2;
    const DenseArgs& d;
    uint32_t K, rows, parts, npass, nst, nu, v, n, g, lob;
    Cursor cn, cc;
    const uint16_t *w0, *w1;  // the unit's rows of the two matrices
    uint32_t wbytes, vw[2], col0;
    UnitInfo cu;  // e: its split
    f32x4 acc[2][NB], sum[2][NB], err[2][NB];

    static constexpr bool kOnce = true;
    WL_MEM static bool unit_end() { return true; }
    WL_MEM UnitInfo unit(uint32_t i) const {
        UnitInfo x{false, 0u, 0u, 0u, 0u};
        if (i >= nu) return x;
        // (the passes of one block of weights side by side on one XCD)
        const PassPart jp = pass_part(blockIdx.x + gridDim.x * i, npass, parts * d.S);
        x.live = true;
        x.part = jp.j / d.S;
        x.e = jp.j % d.S;
        const uint32_t q = d.T / npass, r = d.T % npass;
        x.row0 = jp.part * q + min(jp.part, r);
        x.nt = q + (jp.part < r ? 1u : 0u);
        return x;
    }
    WL_MEM void bind(uint32_t i, AS& A) {
        const UnitInfo x = unit(i);
        A.kd2 = 2u * K;
        const uint16_t* rows3 = (UP ? d.norm3 : d.mid3) + (size_t)x.row0 * 3u * K;
        A.rs = make_rsrc(x.live ? rows3 : nullptr, x.live ? x.nt * 3u * A.kd2 : 0u);
        const uint32_t r0 = 4u * v + g, cg = n ^ (r0 & 15u);
#pragma unroll
        for (uint32_t j = 0; j < 2; j++) {
            const uint32_t m = r0 + 32u * j;
            A.base[j] = m < x.nt ? m * 3u * A.kd2 + 16u * cg : kOOBV;
        }
        col0 = x.e * nst * 128u;
        const uint32_t first = x.part * kRows;
        w0 = !x.live ? nullptr : (UP ? d.gate : d.down) + (size_t)first * K;
        w1 = !x.live ? nullptr : UP ? d.up + (size_t)first * K : w0;
        wbytes = !x.live ? 0u : min(kRows, rows - first) * K * 2u;
    }
    template <int S>
    WL_MEM void dma(const AS& A, uint32_t s, uint32_t j) const {
        const uint32_t h = j % kRB2, pc = j / kRB2, cg = n ^ ((4u * v + g) & 15u), c = col0 + 128u * s;
        dma16<S>(A.rs, (16u * pc + 8u * h + v) * 1024u, c + 8u * cg < K ? A.base[h] : kOOBV, 2u * c + pc * A.kd2);
    }
    // Loads 2i and 2i + 1 of a tile: its first and last eight rows, 64 columns.
    WL_MEM void load(uint32_t s, WB& W, uint32_t j) const {
        const uint32_t t = j / 4u, c = col0 + 128u * s + 64u * (j % 4u / 2u);
        W.w[j] = bld16(make_rsrc(t ? w1 : w0, wbytes), c + 8u * g + 4u * (n & 8u) < K ? vw[t] + (j % 2u) * 16u * K : kOOBV,
                       2u * c);
    }
    // Such a pair -> row n of the tile in lane (n, g): columns 8 g of its first 32
    // in x, of its last 32 in y (lanes n >= 8 of x trade with lanes n < 8 of y).
    WL_MEM static void rows_swap(u32x4& x, u32x4& y) {
#pragma unroll
        for (uint32_t q = 0; q < 4; q++) {
            const int a = (int)x[q], b = (int)y[q];
            x[q] = (uint32_t)__builtin_amdgcn_update_dpp(a, b, 0x128, 0xF, 0xC, false);  // row_ror:8, lanes 8-15
            y[q] = (uint32_t)__builtin_amdgcn_update_dpp(b, a, 0x128, 0xF, 0x3, false);  // lanes 0-7
        }
    }
    WL_MEM void begin(uint32_t i) {
        cu = unit(i);
#pragma unroll
        for (uint32_t t = 0; t < 2; t++)
#pragma unroll
            for (uint32_t m = 0; m < NB; m++) sum[t][m] = err[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // Iteration it: columns 32 (it % 4) of the step, of the third pieces, then the
    // second, then the first: the sums round at the small pieces' size until the
    // last four (error against 64 bits 9.9e-8 at 200 positions; 1.4e-7 in
    // SharedK::comp's order, where all twelve round at the first piece's).
    template <class Next>
    WL_MEM void comp(uint32_t, const uint8_t* sl, WB& W, Next next) {
        auto frag = [&](uint32_t it, uint32_t m) {
            return as_bf16x8(*(const u32x4*)(sl + ((2u - it / 4u) * 64u + m * 16u) * 256u + (lob ^ (64u * (it % 4u)))));
        };
        bf16x8 af[2][NB];
#pragma unroll
        for (uint32_t m = 0; m < NB; m++) af[0][m] = frag(0u, m);
#pragma unroll
        for (uint32_t it = 0; it < 12u; it++) {
            const uint32_t k = it % 4u;
            if (it + 1u < 12u) {
#pragma unroll
                for (uint32_t m = 0; m < NB; m++) af[(it + 1u) & 1u][m] = frag(it + 1u, m);
            }
            if (it == 0u || it == 2u) {
                rows_swap(W.w[k], W.w[k + 1u]);
                rows_swap(W.w[4u + k], W.w[5u + k]);
            }
            next(it, 12u);
#pragma unroll
            for (uint32_t t = 0; t < 2; t++) {
                const bf16x8 bw = as_bf16x8(W.w[4u * t + k]);
#pragma unroll
                for (uint32_t m = 0; m < NB; m++) {
                    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
                    acc[t][m] = mma(bw, af[it & 1u][m], it == 0u ? z : acc[t][m]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (uint32_t t = 0; t < 2; t++)
#pragma unroll
            for (uint32_t m = 0; m < NB; m++)
#pragma unroll
                for (uint32_t i = 0; i < 4; i++) {
                    const float x = sum[t][m][i], y = acc[t][m][i], z = __fadd_rn(x, y), w = __fsub_rn(z, x);
                    sum[t][m][i] = z;
                    err[t][m][i] += __fadd_rn(__fsub_rn(x, __fsub_rn(z, w)), __fsub_rn(y, w));
                }
    }
    WL_MEM float total(uint32_t t, uint32_t m, uint32_t i) const {
        const float x = sum[t][m][i];
        return fabsf(x) < INFINITY ? x + err[t][m][i] : x;
    }
    WL_MEM void finish() {
        const uint32_t ln = opaque_lane(), nn = ln & 15u, gg = ln >> 4;
#pragma unroll
        for (uint32_t m = 0; m < NB; m++) {
            const uint32_t r = 16u * m + nn;
            if constexpr (UP) {
                const uint32_t col = cu.part * kRows + 16u * v + 4u * gg;
                float xs[4];
#pragma unroll
                for (uint32_t i = 0; i < 4; i++) xs[i] = silu_mul(total(0, m, i), total(1, m, i));
                if (r < cu.nt && col < rows) store_pieces4<true>(d.mid3 + (size_t)(cu.row0 + r) * 3u * rows + col, rows, xs);
                __builtin_amdgcn_sched_barrier(0);
            } else {
#pragma unroll
                for (uint32_t t = 0; t < 2; t++) {
                    const uint32_t col = cu.part * kRows + 32u * v + 16u * t + 4u * gg;
                    if (r < cu.nt && col < rows)
                        gst((f32x4*)(d.part + ((size_t)cu.e * d.T + cu.row0 + r) * rows + col), f32x4{total(t, m, 0), total(t, m, 1), total(t, m, 2), total(t, m, 3)});
                }
            }
        }
    }
};
template <bool UP, uint32_t NB>
__global__ void __launch_bounds__(kGT) dgemm_kernel(const DenseArgs d) {
    DenseK<UP, NB> k{d};
    k.K = UP ? d.H : d.DI;
    k.rows = UP ? d.DI : d.H;
    k.parts = cdiv(k.rows, k.kRows);
    k.npass = d.np;
    k.nst = cdiv(cdiv(k.K, 128u), d.S);
    const uint32_t U = k.npass * k.parts * d.S, lane = threadIdx.x & 63u;
    k.nu = U > blockIdx.x ? cdiv(U - blockIdx.x, gridDim.x) : 0u;
    k.n = lane & 15u;
    k.g = lane >> 4;
    k.v = uni(threadIdx.x >> 6);
#pragma unroll
    for (uint32_t t = 0; t < 2; t++)
        k.vw[t] = ((UP ? 16u * k.v : 32u * k.v + 16u * t) + (k.n & 7u)) * k.K * 2u + 16u * k.g + 8u * (k.n & 8u);
    k.lob = k.n * 256u + 16u * (k.g ^ k.n);
    run_units(k);
}
// out = resid + the partial rows' sum, in order.
__global__ void __launch_bounds__(256) dsum_kernel(const DenseArgs d) {
    const uint64_t n = (uint64_t)d.T * d.H / 4u, i = (uint64_t)blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    f32x4 s = gld((const f32x4*)d.part + i);
    for (uint32_t k = 1; k < d.S; k++) s += gld((const f32x4*)d.part + k * n + i);
    if (d.resid) s += gld((const f32x4*)d.resid + i);
    gst((f32x4*)d.out + i, s);
}
