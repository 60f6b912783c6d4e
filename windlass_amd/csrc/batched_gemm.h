// batched_gemm.h — the expert GEMMs of the batched layer (included by
// moe_batched.hip, inside namespace wl).
//
// Every work-group is eight waves with a whole CU (LDS), two per SIMD, so that
// one wave's matrix instructions run while the other is held at a load: issuing
// the loads takes about as long as the matrix instructions (measured at 64-token
// passes with one wave per SIMD and twice the tiles per wave: a step of 2560
// cycles of MFMA took 4576, the loads adding 112 cycles each). A pipeline runs
// units of one form (a token pass of NB row blocks of 16 tokens times a block of
// weight rows, in nst steps of K): the bf16 shared expert (SharedK), then the
// routed passes from four row blocks down to one (QWide, QNarrow). A work-group
// walks its units u = blockIdx.x + G i of each pipeline. Activations arrive in
// LDS by DMA (buffer_load ... lds), weights in registers. The weights are the
// matrix instructions' A operand (its rows), the tokens its columns: a lane then
// holds four consecutive outputs of one token, stored as 16 bytes.
#pragma once

constexpr uint32_t kSlotB = 48u << 10;
constexpr uint32_t kOOBV = 0x80000000u;  // a lane offset past every array (they stay below 2 GB)
// Three slots of activations, separate LDS objects so that the compiler's own
// waits for DMA-written LDS stay per slot.
__shared__ __align__(16) uint8_t g_slot0[kSlotB];
__shared__ __align__(16) uint8_t g_slot1[kSlotB];
__shared__ __align__(16) uint8_t g_slot2[kSlotB];
template <int S>
WL_DEV uint8_t* slot() {
    return S == 0 ? g_slot0 : S == 1 ? g_slot1 : g_slot2;
}
template <int S>
WL_DEV void dma16(rsrc_t rs, uint32_t lds, uint32_t voff, uint32_t soff) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (__attribute__((address_space(3))) void*)(slot<S>() + lds), 16u, voff,
                                             soff, 0, 0);
}
// s_waitcnt vmcnt(N) (expcnt, lgkmcnt not waited on), barrier.
template <uint32_t N>
WL_DEV void step_barrier() {
    static_assert(N < 64u, "vmcnt is 6 bits");
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt((N & 15u) | ((N >> 4) << 14) | 0x0F70u);
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}
// Between two pipelines of one kernel: every load and DMA of the first has
// landed and every wave is done with its slots.
WL_DEV void pipeline_drain() { step_barrier<0>(); }

// A unit: a token pass (of the batch, or an expert's) and its block of weight
// rows.
struct UnitInfo {
    bool live;
    uint32_t e, part, nt, row0;
    uint32_t m0 = 0u, m1 = 4u;  // its slices (gate/up of small passes; others have all four)
};
// Which units are a work-group's. The units of a kernel stand in one row, position s:
// the shared expert's from 0, then the routed passes'. Position s < G is work-group
// s's, a later one work-group (s + skip) % G's: skip work-groups, those of the shared
// expert's units, go without one of the second round.
struct Places {
    uint32_t base, s0, s1;  // the pipeline's first position, the work-group's first two there
    WL_MEM static Places from(uint32_t base, uint32_t skip) {
        const uint32_t G = gridDim.x, b = blockIdx.x, l = b >= skip ? G + b - skip : 2u * G + b - skip;
        if (base <= b) return Places{base, b, l};
        const uint32_t s0 = l + (base > l ? cdiv(base - l, G) : 0u) * G;
        return Places{base, s0, s0 + G};
    }
    WL_MEM uint32_t place(uint32_t i) const { return i == 0u ? s0 : s1 + (i - 1u) * gridDim.x; }
    WL_MEM uint32_t count(uint32_t end) const {  // those below position end
        return s0 >= end ? 0u : s1 >= end ? 1u : 1u + cdiv(end - s1, gridDim.x);
    }
};

// ---- pipeline ------------------------------------------------------------------------
// Position of a stream in the units' steps: my unit i (of a pipeline whose units may
// run their steps twice, that run), its step s.
struct Cursor {
    uint32_t i, s;
};
WL_DEV bool advance(Cursor& c, uint32_t nst) {
    if (++c.s < nst) return false;
    c.s = 0;
    c.i++;
    return true;
}
// The steps of a work-group's units form one flat sequence z. A pipeline has one
// form of unit, so that every value keeps its registers through the loop (with
// forms chosen per unit the compiler moved the loads in flight between registers
// at the units' ends, which waits for them). The loads run two steps ahead
// of the compute, through the units' ends. Step z: this wave's loads of the step,
// issued two steps ago, have landed ("at most the loads of one step
// outstanding": they complete in issue order) and the waves have met, so every
// wave's activations are there and every wave is done with step z - 1, whose slot
// and registers take the loads of step z + 2; these go out evenly between the
// matrix instructions of step z (all at its start: 7 to 18 % slower per call). The loop runs whole rounds
// of three steps; the loads of the steps past the last unit are out of range
// (zeros) and what they compute is not stored.
template <int S, class Kn>
WL_DEV void unit_step(Kn& k, typename Kn::AS& A, typename Kn::WB& cur, typename Kn::WB& nxt) {
    constexpr uint32_t L = Kn::kDmas + Kn::kLoads;
    constexpr int SN = (S + 2) % 3;
    step_barrier<L>();
    if (advance(k.cn, k.nst)) k.bind(k.cn.i, A);
    const uint32_t sn = k.cn.s;
    // called n times over a step (it = 0 .. n - 1)
    auto next = [&](uint32_t it, uint32_t n) {
#pragma unroll
        for (uint32_t j = 0; j < L; j++) {
            if (j * n / L != it) continue;
            if (j < Kn::kDmas) k.template dma<SN>(A, sn, j);
            else k.load(sn, nxt, j - Kn::kDmas);
        }
    };
    __builtin_amdgcn_sched_barrier(0);
    k.comp(k.cc.s, slot<S>(), cur, next);
    if (advance(k.cc, k.nst) && k.unit_end()) {
        if (Kn::kOnce ? k.cc.i <= k.nu : k.cu.live) k.finish();
        k.begin(k.cc.i);
    }
}
template <class Kn>
WL_DEV void run_units(Kn& k) {
    if (k.nu == 0u) return;
    const uint32_t Z = k.nu * k.nst;
    typename Kn::AS A;
    typename Kn::WB B0, B1, B2;
    k.cn = k.cc = Cursor{0u, 0u};
    k.begin(0u);
    k.bind(0u, A);
#pragma unroll
    for (uint32_t j = 0; j < Kn::kDmas; j++) k.template dma<0>(A, 0u, j);
#pragma unroll
    for (uint32_t j = 0; j < Kn::kLoads; j++) k.load(0u, B0, j);
    if (advance(k.cn, k.nst)) k.bind(k.cn.i, A);
#pragma unroll
    for (uint32_t j = 0; j < Kn::kDmas; j++) k.template dma<1>(A, k.cn.s, j);
#pragma unroll
    for (uint32_t j = 0; j < Kn::kLoads; j++) k.load(k.cn.s, B1, j);
    auto round = [&]() {
        unit_step<0>(k, A, B0, B2);
        unit_step<1>(k, A, B1, B0);
        unit_step<2>(k, A, B2, B1);
    };
    // (counted where it can be: with the other loop the dense layers took 1 to 5 %
    // longer)
    if constexpr (Kn::kOnce) {
#pragma unroll 1
        for (uint32_t z = 0; z < Z; z += 3u) round();
    } else {
#pragma unroll 1
        do round();
        while (k.cu.live);
    }
}

// ---- outputs ---------------------------------------------------------------------------
// The epilogues pass the lane through opaque_lane, so the compiler cannot hoist
// their per-row addresses out of the step loop.
WL_DEV uint32_t opaque_lane() {
    uint32_t l = threadIdx.x & 63u;
    asm volatile("" : "+v"(l));
    return l;
}
// SwiGLU of two gate/up tiles (rows 0-7 gate, 8-15 the matching up rows; lane
// (n, g) holds rows 4g .. 4g + 3 of token n): one swap per value brings the gate
// values of both tiles together and their up values, so lane (n, g) gets columns
// 4 (g % 2) .. +4 of tile g / 2 for token n.
WL_DEV f32x4 swiglu_pair(const f32x4& a, const f32x4& b) {
    f32x4 r;
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) {
        uint32_t gt, up;
        swap32(__float_as_uint(a[i]), __float_as_uint(b[i]), gt, up);
        r[i] = silu_mul(__uint_as_float(gt), __uint_as_float(up));
    }
    return r;
}

// ---- shared expert (bf16) ----------------------------------------------------------------
// Three bf16 pieces of each activation (x = p0 + p1 + p2 to f32 precision)
// through v_mfma_f32_16x16x32_bf16; the first piece and the other two sum in
// accumulators of their own, and with NT = 1 the first piece's are added to the
// sums at every step (a long chain of matrix instructions rounds more often). Unit: a pass of the batch (its tokens split evenly
// over cdiv(T, 64) passes, NB row blocks) x 8 waves x NT tiles. UP: tiles of 8
// gate and 8 up rows (native sgu chunks: lane (n, g) row n, columns [32 kt + 8
// g, +8)), K = H, SwiGLU values as pieces to smid3. Otherwise tiles of 16 output
// rows (native sdn: 16 bytes = columns [8T, +8) of a row, lane (n, g) tile 4 kt +
// g of row n), K = SI, f32 rows to shout. A step is 128 columns. NT = 1: small
// batches, more units; NT = 2: a fragment feeds two tiles.
//
// Slot: row R = 64 pc + m (token m, piece pc) of 256 bytes, its 16-byte group p
// holding columns [k0 + 8 (p ^ (R & 15)), +8), so that the 16 rows a fragment
// reads at one column fall in 16 different bank groups. A DMA of wave v writes rows
// 64 pc + 32 j + r0, r0 = 4 v + (lane >> 4) < 32, of piece pc (j = 0, 1).
struct AStreamS {
    rsrc_t rs;
    uint32_t base[2], kd2;  // lane byte offsets of the tokens r0 + 32 j (kOOBV: none), bytes per piece row
};
template <bool UP, uint32_t NT, uint32_t NB>
struct SharedK {
    using AS = AStreamS;
    struct WB {
        u32x4 w[4 * NT];
    };
    static constexpr uint32_t kLoads = 4 * NT, kRB2 = (NB + 1) / 2, kDmas = 3 * kRB2;
    const DecodeArgs& a;
    const BatchArgs& b;
    uint32_t H, SI, nkt, parts, npass, nst, nu, v, n, g;
    Cursor cn, cc;  // positions of the loads and of the compute
    // weight stream: the block, kept as a pointer and a size (a buffer resource
    // held in a struct has gone through scratch, its loads per-lane loops)
    const uint8_t* wbase;
    uint32_t wbytes, wpart, vw[UP ? 1 : NT], lob;
    UnitInfo cu;
    static constexpr bool kSum = NT == 1u;
    f32x4 acc[NT][NB][2], sum[kSum ? NT : 1][kSum ? NB : 1];

    static constexpr bool kOnce = true;  // its units run their steps once
    WL_MEM static bool unit_end() { return true; }
    WL_MEM UnitInfo unit(uint32_t i) const {
        UnitInfo x{false, 0u, 0u, 0u, 0u};
        if (i >= nu) return x;
        const PassPart jp = pass_part(blockIdx.x + gridDim.x * i, parts, npass);
        x.live = true;
        x.part = jp.part;
        const uint32_t q = b.T / npass, r = b.T % npass;
        x.row0 = jp.j * q + min(jp.j, r);
        x.nt = q + (jp.j < r ? 1u : 0u);
        return x;
    }
    // Unit i's streams (i >= nu: nothing to load).
    WL_MEM void bind(uint32_t i, AS& A) {
        const UnitInfo x = unit(i);
        A.kd2 = 2u * (UP ? H : SI);
        A.rs = make_rsrc(x.live ? (UP ? b.norm3 : b.smid3) : nullptr, x.live ? b.T * 3u * A.kd2 : 0u);
        const uint32_t r0 = 4u * v + g, cg = n ^ (r0 & 15u);
#pragma unroll
        for (uint32_t j = 0; j < 2; j++) {
            const uint32_t m = r0 + 32u * j;
            A.base[j] = m < x.nt ? (x.row0 + m) * 3u * A.kd2 + 16u * cg : kOOBV;
        }
        const NativeShared NS = NativeShared::make(H, SI);
        wpart = x.part;
        wbase = !x.live ? nullptr : a.sh_native + (UP ? NS.sgu : NS.sdn);
        wbytes = !x.live ? 0u : (uint32_t)(UP ? NS.sdn - NS.sgu : NS.total - NS.sdn);
        if (!UP) {
#pragma unroll
            for (uint32_t t = 0; t < NT; t++)
                vw[UP ? 0 : t] = (g * H + min(16u * (NT * (kGW * x.part + v) + t) + n, H - 1u)) * 16u;
        }
    }
    template <int S>
    WL_MEM void dma(const AS& A, uint32_t s, uint32_t j) const {
        const uint32_t h = j % kRB2, pc = j / kRB2;
        dma16<S>(A.rs, (16u * pc + 8u * h + v) * 1024u, A.base[h], 256u * s + pc * A.kd2);
    }
    WL_MEM void load(uint32_t s, WB& W, uint32_t j) const {
        const rsrc_t rs = make_rsrc(wbase, wbytes);
        const uint32_t t = j / 4u, k = j % 4u;
        if (UP) W.w[j] = bld16(rs, vw[0], ((NT * (kGW * wpart + v) + t) * nkt + 4u * s + k) * 1024u);
        else W.w[j] = bld16(rs, vw[UP ? 0 : t], (16u * s + 4u * k) * H * 16u);
    }
    WL_MEM void begin(uint32_t i) {
        cu = unit(i);
        const f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (uint32_t t = 0; t < NT; t++)
#pragma unroll
            for (uint32_t m = 0; m < NB; m++) {
                acc[t][m][0] = acc[t][m][1] = z;
                if constexpr (kSum) sum[t][m] = z;
            }
    }
    // Iteration it = 3 k + pc: plane pc of k step k (columns 32 k + 8 g of the
    // step, group cg = 4 k + g: lane offset lob ^ 64 k) against the tiles; the
    // next iteration's NB fragments are read while this one's MFMAs run.
    template <class Next>
    WL_MEM void comp(uint32_t, const uint8_t* sl, WB& W, Next next) {
        auto frag = [&](uint32_t it, uint32_t m) {
            return as_bf16x8(*(const u32x4*)(sl + ((it % 3u) * 64u + m * 16u) * 256u + (lob ^ (64u * (it / 3u)))));
        };
        bf16x8 af[2][NB];
#pragma unroll
        for (uint32_t m = 0; m < NB; m++) af[0][m] = frag(0u, m);
#pragma unroll
        for (uint32_t it = 0; it < 12u; it++) {
            const uint32_t k = it / 3u, pc = it % 3u;
            if (it + 1u < 12u) {
#pragma unroll
                for (uint32_t m = 0; m < NB; m++) af[(it + 1u) & 1u][m] = frag(it + 1u, m);
            }
            next(it, 12u);
#pragma unroll
            for (uint32_t t = 0; t < NT; t++) {
                const bf16x8 bw = as_bf16x8(W.w[4u * t + k]);
#pragma unroll
                for (uint32_t m = 0; m < NB; m++) {
                    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
                    f32x4& c = acc[t][m][pc ? 1 : 0];
                    c = mma(bw, af[it & 1u][m], kSum && it == 0u ? z : c);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (kSum) {
#pragma unroll
            for (uint32_t t = 0; t < NT; t++)
#pragma unroll
                for (uint32_t m = 0; m < NB; m++) sum[t][m] += acc[t][m][0];
        }
    }
    WL_MEM f32x4 total(uint32_t t, uint32_t m) const {
        if constexpr (kSum) return sum[t][m] + acc[t][m][1];
        else return acc[t][m][0] + acc[t][m][1];
    }
    WL_MEM void finish() {
        const uint32_t ln = opaque_lane(), nn = ln & 15u, gg = ln >> 4;
        const uint32_t T0 = NT * (kGW * cu.part + v);
        if constexpr (UP) {
            // pairs of tiles, or of row blocks of the one tile
            constexpr uint32_t NP = NT == 1u ? (NB + 1u) / 2u : NB;
#pragma unroll
            for (uint32_t m = 0; m < NP; m++) {
                const uint32_t m0 = NT == 1u ? 2u * m : m, m1 = NT == 1u ? (2u * m + 1u < NB ? 2u * m + 1u : m0) : m;
                const f32x4 x = swiglu_pair(total(0u, m0), total(NT - 1u, m1));
                const float xs[4] = {x[0], x[1], x[2], x[3]};
                const uint32_t r = 16u * (NT == 1u ? 2u * m + (gg >> 1) : m) + nn;
                const uint32_t col = 8u * T0 + (NT == 1u ? 4u * (gg & 1u) : 4u * gg);
                if (r < cu.nt) store_pieces4(b.smid3 + (size_t)(cu.row0 + r) * 3u * SI + col, SI, xs);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
#pragma unroll
            for (uint32_t m = 0; m < NB; m++) {
                const uint32_t r = 16u * m + nn;
#pragma unroll
                for (uint32_t t = 0; t < NT; t++) {
                    const uint32_t row = 16u * (T0 + t) + 4u * gg;
                    if (r < cu.nt && row < H) gst((f32x4*)(b.shout + (size_t)(cu.row0 + r) * H + row), total(t, m));
                }
            }
        }
    }
};
// Its units are the first; returns their count.
template <bool UP, uint32_t NT, uint32_t NB>
WL_DEV uint32_t run_shared(const DecodeArgs& a, const BatchArgs& b) {
    SharedK<UP, NT, NB> k{a, b};
    k.H = a.H;
    k.SI = a.SI;
    k.nkt = a.H / 32u;
    k.parts = UP ? a.SI / (8u * kGW * NT) : cdiv(a.H, 16u * kGW * NT);
    k.npass = cdiv(b.T, 64u);
    k.nst = (UP ? a.H : a.SI) / 128u;
    const uint32_t U = k.npass * k.parts, lane = threadIdx.x & 63u;
    k.nu = U > blockIdx.x ? cdiv(U - blockIdx.x, gridDim.x) : 0u;
    k.n = lane & 15u;
    k.g = lane >> 4;
    k.v = uni(threadIdx.x >> 6);
    if (UP) k.vw[0] = 16u * lane;
    k.lob = k.n * 256u + 16u * (k.g ^ k.n);
    run_units(k);
    return U;
}
// (More than two passes: the largest has at least 43 tokens, so three row
// blocks or four.)
template <bool UP>
WL_DEV uint32_t run_shared_expert(const DecodeArgs& a, const BatchArgs& b) {
    if (b.flags & (kBatchNoShared | kBatchShared4)) return 0u;
    const uint32_t np = cdiv(b.T, 64u), nb = cdiv(cdiv(b.T, np), kRB);
    if (np > 2u) return nb == 3u ? run_shared<UP, 2, 3>(a, b) : run_shared<UP, 2, 4>(a, b);
    switch (nb) {
        case 1: return run_shared<UP, 1, 1>(a, b);
        case 2: return run_shared<UP, 1, 2>(a, b);
        case 3: return run_shared<UP, 1, 3>(a, b);
        default: return run_shared<UP, 1, 4>(a, b);
    }
}

// ---- routed experts (MXFP4) ---------------------------------------------------------------
// On rows quantised by q6.h.
//
// w: 16 weight rows of 128 columns in MXFP4, x: one piece of 16 tokens; byte ow
// of sw and byte ox of sx are the lane's block scales (compile-time constants
// after unrolling).
WL_DEV f32x4 mmq(u32x4 w, i32x8 x, f32x4 c, uint32_t ow, uint32_t sw, uint32_t ox, uint32_t sx) {
    const i32x8 A = {(int)w.x, (int)w.y, (int)w.z, (int)w.w, 0, 0, 0, 0};
#define WL_MMQ(i, j) \
    case 4 * i + j: return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(A, x, c, 4, 2, i, (int)sw, j, (int)sx)
    switch (4u * ow + ox) {
        WL_MMQ(0, 0); WL_MMQ(0, 1); WL_MMQ(0, 2); WL_MMQ(0, 3);
        WL_MMQ(1, 0); WL_MMQ(1, 1); WL_MMQ(1, 2); WL_MMQ(1, 3);
        WL_MMQ(2, 0); WL_MMQ(2, 1); WL_MMQ(2, 2); WL_MMQ(2, 3);
        WL_MMQ(3, 0); WL_MMQ(3, 1); WL_MMQ(3, 2); WL_MMQ(3, 3);
    }
#undef WL_MMQ
    return c;
}
// A staged k tile of 16 rows: kilobyte 2 u + h holds units 8 u .. 8 u + 7 of rows
// 8 h .. 8 h + 7, 128 bytes a row, unit c in its 16-byte place c ^ q_swizzle(row),
// so that the 16 rows of a fragment read fall in different banks.
WL_DEV uint32_t q_swizzle(uint32_t n) { return (n & 7u) ^ (n >> 3); }
// The lane's offsets of unit g of row n, and of its 8 bytes of unit g / 2.
WL_DEV uint32_t q_lo16() {
    const uint32_t lane = threadIdx.x & 63u, n = lane & 15u, g = lane >> 4;
    return 1024u * (n >> 3) + 128u * (n & 7u) + 16u * (g ^ q_swizzle(n));
}
WL_DEV uint32_t q_lo8() {
    const uint32_t lane = threadIdx.x & 63u, n = lane & 15u, g = lane >> 4;
    return 1024u * (n >> 3) + 128u * (n & 7u) + 16u * ((g >> 1) ^ q_swizzle(n)) + 8u * (g & 1u);
}
// From the lane's offset lo of unit i (< 4 for c a multiple of 4, < 2 for an even
// c): that of unit c + i.
WL_DEV const uint8_t* q_at(const uint8_t* tile, uint32_t c, uint32_t lo) {
    return tile + 2048u * (c / 8u) + (lo ^ (16u * (c % 8u)));
}
// Piece p of the tile.
WL_DEV i32x8 q_frag(const uint8_t* tile, uint32_t p, uint32_t lo16, uint32_t lo8) {
    const u32x4 h = *(const u32x4*)q_at(tile, 4u * p, lo16);
    const u32x2 l = *(const u32x2*)q_at(tile, 4u * kQP + 2u * p, lo8);
    return i32x8{(int)h.x, (int)h.y, (int)h.z, (int)h.w, (int)l.x, (int)l.y, 0, 0};
}
WL_DEV u32x2 q_scales(const uint8_t* tile, uint32_t lo8) {
    return *(const u32x2*)q_at(tile, 6u * kQP, lo8);
}
// Two chunks of 64 columns of a row pair (lane (n, g): row 32 q + n + 16 (g >>
// 1), block g & 1) -> 128 columns of each of its halves, in place.
WL_DEV void pair_swap(u32x4& x, u32x4& y) {
#pragma unroll
    for (uint32_t d = 0; d < 4; d++) {
        uint32_t lo, hi;
        swap32(x[d], y[d], lo, hi);
        x[d] = lo;
        y[d] = hi;
    }
}

// MB row blocks, KT k tiles per step: the slot holds tile (q, m), number MB q + m.
// A DMA of a tile fills one of its kilobytes: 128 bytes of each of eight rows, a
// row by eight lanes next to each other (lane l: row 8 h + l / 8). Wave v takes
// kilobyte v of every tile, then one of the two left over of tile v / 2: kilobyte 8 +
// v % 2 (past the tiles: out of range, into the slot's end). (Lanes that took 64 bytes of each of 16 rows, every
// quarter wave 16 cache lines: 1000 tokens 1588 us a call, now 1556; 333 of hidden
// 2944 309, 305; 7, 64 and 4096 the same within 0.4 %.) Absent rows, k tiles past the row's end and units past the record
// land as zeros (zero scales too: their products are zero).
template <uint32_t MB>
struct AStreamQ {
    rsrc_t rs, rs1;  // (rs1: of further pieces beside the records)
    // lane byte offsets of the lane's units of its rows (left: of its left-over
    // unit), k tiles of a row, bytes of a record
    uint32_t base[MB], left, nk, rec;
};
// What the pipelines share: the layer's tables, the rows of a pass, the
// epilogues. UP: gate/up of the routed experts, K = H, slices of 64 rows (tiles of
// 8 gate and 8 up rows), SwiGLU values to midf.
// Otherwise down, K = I, row pairs (rows 32 q + n and + 16), to expout. A unit
// is four slices, or 16 row pairs: four tiles per wave (tile 8 sl + v of slice
// sl, row pairs 2 v and 2 v + 1 of the 16), as the native block's batched scale
// words are laid out. NB row blocks, KT k tiles per step.
// FOLD (NB = 1): a row's further pieces stand beside its record, as a second row block.
template <bool UP, uint32_t NB, uint32_t KT, bool FOLD = false>
struct QBase {
    static constexpr uint32_t MB = FOLD ? 2u : NB;  // row blocks staged
    using AS = AStreamQ<MB>;
    static constexpr uint32_t P = kQP, NG = (kQUnits + 3u) / 4u;  // groups of a record
    static constexpr uint32_t kTiles = MB * KT, kTileB = 1024u * NG, kDmas = kTiles + 1u;
    static_assert(NG == 10u && kTiles <= 4u, "ten groups of at most four tiles");
    static_assert(kTileB * kTiles + 8192u <= kSlotB, "a step's tiles fit a slot");
    const DecodeArgs& a;
    const BatchArgs& b;
    uint32_t H, I, E, K, nk, S, nq, parts, nst, nst2, nu, v, lane;
    Places pl;
    uint32_t tail, cut;  // units from position tail on are cut into 1 << cut
    PassTab pt;
    const uint8_t* const* stab;
    NativeLayout NL;
    Cursor cn, cc;  // positions of the loads and of the compute
    const uint8_t* wbase;  // the weight stream's block and size (see SharedK)
    uint32_t wbytes, wpart, wm0, wm1, vw, vs, lo8, lo16;
    UnitInfo cu, un;     // the unit computed, the unit whose loads go out
    // any row of the call has further pieces; the positions of these units among the
    // work-group's, whether they run twice and are in their second run
    bool any;
    uint32_t ci, ni;
    bool ctwice, csecond, ntwice, nsecond;
    const uint16_t* tt;  // UP: the token table, or the tokens of all entries where this kernel grouped them

    WL_MEM UnitInfo unit(uint32_t i) const {
        UnitInfo x{false, 0u, 0u, 0u, 0u};
        if (i >= nu) return x;
        uint32_t s = pl.place(i);
        if (s >= tail) {
            const uint32_t w = 4u >> cut, p = (s - tail) & ((1u << cut) - 1u);
            s = tail + ((s - tail) >> cut);
            x.m0 = p * w;
            x.m1 = x.m0 + w;
        }
        const PassPart jp = pass_part(s - pl.base, parts, pt.n);
        const Pass ps = pass_at(pt, E, jp.j);
        x.live = true;
        x.part = jp.part;
        x.e = ps.e;
        x.nt = ps.nt;
        x.row0 = ps.c0;
        return x;
    }
    // The activation row of row r (< nt) of unit i.
    WL_MEM uint32_t row_of(const UnitInfo& x, uint32_t i, uint32_t r) const {
        if (!UP) return x.row0 + r;
        if (x.e == a.E) return x.row0 + r - b.T * K;
        return b.group ? (uint32_t)tt[x.row0 + min(r, x.nt - 1u)] : table_token(tt, b.tcap, kRB * NB, i, r, x.nt);
    }
    // A unit with a row of further pieces runs its steps twice: on the records, then
    // on the further pieces.
    WL_MEM bool twice(const UnitInfo& x, uint32_t i) const {
        if (FOLD || !any || !x.live) return false;
        static_assert(kRB * NB <= 64u, "a lane per row");
        const bool has = lane < x.nt && gld((UP ? b.more_up : b.more_dn) + row_of(x, i, min(lane, x.nt - 1u))) != 0u;
        return __builtin_amdgcn_ballot_w64(has) != 0u;
    }
    // (called once for each run, in order)
    WL_MEM void bind(uint32_t run, AS& A) {
        nsecond = run > 0u && ntwice && !nsecond;
        if (!nsecond) {
            ni = run == 0u ? 0u : ni + 1u;
            un = unit(ni);
            ntwice = twice(un, ni);
        }
        const uint32_t i = ni;
        const bool more = nsecond;
        const UnitInfo x = un;
        const uint8_t* blk = x.live ? uni_ptr(stab[x.e]) : nullptr;
        wbase = blk;
        wbytes = blk ? (uint32_t)NL.total : 0u;
        wpart = x.part;
        wm0 = x.m0;
        wm1 = x.m1;
        const uint32_t kd = UP ? H : I, n = 8u * (v & 1u) + lane / 8u, c8 = lane % 8u ^ q_swizzle(n);
        const uint32_t nrow = UP ? b.T : b.T * (K + ((b.flags & kBatchShared4) ? 1u : 0u));
        const uint32_t rec = (uint32_t)q6_row_bytes(kd), ext = (uint32_t)q6_more_bytes(kd);
        auto array = [&](bool lo) {
            const uint8_t* rows = UP ? (const uint8_t*)b.norm : lo ? b.mid6x : b.mid6;
            return make_rsrc(x.live ? rows : nullptr, x.live ? nrow * (UP ? rec + ext : lo ? ext : rec) : 0u);
        };
        A.rs = array(more);
        if (FOLD) A.rs1 = array(true);
        A.nk = x.live ? nk : 0u;
        A.rec = more ? kQMore : kQRecord;
        // the lane's unit c of its row of block m
        auto row_at = [&](uint32_t m, uint32_t c) {
            const bool lo = more || (FOLD && m == 1u);
            const uint32_t r = FOLD ? n : kRB * m + n;
            const uint32_t row = x.live ? row_of(x, i, r) : 0u;
            bool has = r < x.nt && c < kQUnits;
            if (lo) {
                has = has && gld((UP ? b.more_up : b.more_dn) + row) != 0u && q6_more_unit(c) != ~0u;
                c = q6_more_unit(c);
            }
            return has ? row * (UP ? rec + ext : lo ? ext : rec) + (UP && lo ? rec : 0u) + 16u * c : kOOBV;
        };
#pragma unroll
        for (uint32_t m = 0; m < MB; m++) A.base[m] = row_at(m, 8u * (v / 2u) + c8);
        A.left = v / 2u < kTiles ? row_at(v / 2u % MB, 32u + c8) : kOOBV;
    }
    template <int SL>
    WL_MEM void dma(const AS& A, uint32_t s, uint32_t j) const {
        // (wave v's left-over units are those of tile v / 2)
        const uint32_t t = j < kTiles ? j : v / 2u, k = s * KT + t / MB;
        const bool lo = FOLD && t % MB == 1u;
        const uint32_t dst = j < kTiles ? j * kTileB + v * 1024u
                             : t < kTiles ? t * kTileB + (8u + v % 2u) * 1024u : kTiles * kTileB + v * 1024u;
        dma16<SL>(lo ? A.rs1 : A.rs, dst, k >= A.nk ? kOOBV : j < kTiles ? A.base[j % MB] : A.left,
                  k * (lo ? kQMore : A.rec));
    }
    static constexpr bool kOnce = FOLD;
    WL_MEM bool unit_end() {
        csecond = ctwice && !csecond;
        return !csecond;
    }
    WL_MEM void begin_unit(uint32_t run) {
        ci = run == 0u ? 0u : ci + 1u;
        csecond = false;
        if (nst > 1u && run > 0u) {  // (the loads are two steps ahead)
            cu = un;
            ctwice = ntwice;
        } else {
            cu = unit(ci);
            ctwice = twice(cu, ci);
        }
        if (cu.live && stab[cu.e] == nullptr && threadIdx.x == 0) raise_error(a.sync, SyncMap::make(), E_NOT_RESIDENT, 0u);  // no waits in this path: epoch 0 aborts nothing
    }
    // The four slices of row block m, two at a time.
    template <class D>
    WL_MEM void put_up(uint32_t m, D d) const {
        const uint32_t ln = opaque_lane(), r = kRB * m + (ln & 15u), gg = ln >> 4;
        float* o = b.midf + (size_t)(cu.row0 + r) * b.ldm + 8u * v + 4u * (gg & 1u);
#pragma unroll
        for (uint32_t i = 0; i < 4; i += 2) {
            const uint32_t sl = cu.part * 4u + i + (gg >> 1);
            const f32x4 x = swiglu_pair(d(i), d(i + 1u));
            const uint32_t m = i + (gg >> 1);
            if (r < cu.nt && sl < S && m >= cu.m0 && m < cu.m1) gst((f32x4*)(o + sl * kSlice), x);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    WL_MEM void put_down(const f32x4& d, uint32_t m, uint32_t q, uint32_t h) const {
        const uint32_t ln = opaque_lane(), r = kRB * m + (ln & 15u);
        if (r < cu.nt && q < nq) gst((f32x4*)(b.expout + (size_t)(cu.row0 + r) * b.ldm + 32u * q + 16u * h + 4u * (ln >> 4)), d);
    }
};

// Passes of one or two row blocks: bound by the weight stream (a step is 64 KB
// of weights against at most 3600 cycles of MFMA per SIMD); a step has 256
// columns: per wave 8 chunks of 1 KB and the batched scale word (bgus, bdns). UP:
// 4 slices x 2 k tiles; down: 4 slices of 64 columns x 2 row pairs. The first piece and the
// others sum in accumulators of their own; in passes of one row block the first
// piece's are added to the sums at every step in f32 (matrix instructions that
// add into a large sum round it more coarsely). With FOLD a call with further pieces
// reads the weights of its small passes once (a second run of their steps: 7 and 64 tokens with
// outliers in every one 299 and 832 us); a pass without them gives the same bits.
template <bool UP, uint32_t NB, bool FOLD = false>
struct QNarrow : QBase<UP, NB, 2, FOLD> {
    using QB = QBase<UP, NB, 2, FOLD>;
    using QB::P;
    using QB::MB;
    struct WB {
        u32x4 w[8];
        uint32_t s[2];
    };
    static constexpr uint32_t kLoads = 9;
    static constexpr bool kSum = NB == 1u;
    f32x4 acc[4][NB][2], sum[kSum ? 4 : 1];

    WL_MEM QNarrow(const DecodeArgs& a_, const BatchArgs& b_) : QB{a_, b_} {}
    WL_MEM void load(uint32_t s, WB& W, uint32_t j) const {
        const rsrc_t rs = make_rsrc(this->wbase, this->wbytes);
        if (j == 8u) return bld8(rs, this->vs, (this->wpart * 8u * this->nst2 + s) * 512u, W.s);
        uint32_t ch;
        if (UP) ch = min(this->wpart * 4u + j / 2u, this->S - 1u) * 8u * this->nk + min(2u * s + j % 2u, this->nk - 1u);
        else ch = min(4u * s + j / 2u, 2u * this->nk - 1u) * this->nq + min(16u * this->wpart + 2u * this->v + j % 2u, this->nq - 1u);
        const bool has = !UP || NB > 1u || (j / 2u >= this->wm0 && j / 2u < this->wm1);
        W.w[j] = bld16_nt(rs, has ? this->vw : kOOBV, ch * 1024u);
    }
    WL_MEM void begin(uint32_t i) {
        this->begin_unit(i);
        const f32x4 z = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (uint32_t t = 0; t < 4; t++) {
#pragma unroll
            for (uint32_t m = 0; m < NB; m++) acc[t][m][0] = acc[t][m][1] = z;
            if (kSum) sum[t] = z;
        }
    }
    // Operands it in this order: piece p of block m of k tile q, it = (P q + p) NB + m
    // (FOLD: after a k tile's six pieces its further ones); each runs against the wave's
    // weight tiles while the two after it are read.
    template <class Next>
    WL_MEM void comp(uint32_t, const uint8_t* sl, WB& W, Next next) {
        constexpr uint32_t NQ = FOLD ? P + kQX : P * NB, N = 2u * NQ, AH = 2u;
        i32x8 af[AH + 1u];
        u32x2 sa[MB];
        uint32_t sx = 0u, sy = 0u;
        const uint32_t lo16 = this->lo16;
        auto tile = [&](uint32_t q, uint32_t m) { return sl + (q * MB + m) * QB::kTileB; };
        auto block = [](uint32_t it) { return FOLD ? (it % NQ >= P ? 1u : 0u) : it % NB; };
        auto piece = [](uint32_t it) { return FOLD ? (it % NQ >= P ? it % NQ - P : it % NQ) : it / NB % P; };
        auto frag = [&](uint32_t it) { return q_frag(tile(it / NQ, block(it)), piece(it), lo16, this->lo8); };
#pragma unroll
        for (uint32_t it = 0; it < AH; it++) af[it] = frag(it);
#pragma unroll
        for (uint32_t it = 0; it < N; it++) {
            const uint32_t m = block(it), p = piece(it), q = it / NQ;
            if (it % NQ == 0u) {
#pragma unroll
                for (uint32_t i = 0; i < MB; i++) sa[i] = q_scales(tile(q, i), this->lo8);
                if (!UP) {
#pragma unroll
                    for (uint32_t h = 0; h < 2; h++) pair_swap(W.w[4u * q + h], W.w[4u * q + 2u + h]);
                    swap32(W.s[q], W.s[q] >> 16, sx, sy);
                }
            }
            if (it + AH < N) af[(it + AH) % (AH + 1u)] = frag(it + AH);
            next(it, N);
#pragma unroll
            for (uint32_t t = 0; t < 4; t++) {
                // UP: slice t; down: row pair t % 2, half t / 2
                const uint32_t ow = UP ? 2u * (t & 1u) + q : t & 1u;
                const uint32_t sw = UP ? W.s[t >> 1] : (t & 2u) ? sy : sx;
                const u32x4 w = W.w[UP ? 2u * t + q : 4u * q + t];
                const f32x4 z = {0.f, 0.f, 0.f, 0.f};
                const bool first = p == 0u && !(FOLD && m == 1u);
                f32x4& c = acc[t][FOLD ? 0u : m][first ? 0u : 1u];
                c = mmq(w, af[it % (AH + 1u)], kSum && first && q == 0u ? z : c, ow, sw, p & 3u, p < 4u ? sa[m].x : sa[m].y);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (kSum) {
#pragma unroll
            for (uint32_t t = 0; t < 4; t++) sum[t] += acc[t][0][0];
        }
    }
    WL_MEM void finish() {
#pragma unroll
        for (uint32_t m = 0; m < NB; m++) {
            auto d = [&](uint32_t t) {
                if constexpr (kSum) return sum[t] + acc[t][0][1];
                else return acc[t][m][0] + acc[t][m][1];
            };
            if constexpr (UP) {
                this->put_up(m, d);
            } else {
#pragma unroll
                for (uint32_t t = 0; t < 4; t++) this->put_down(d(t), m, this->cu.part * 16u + 2u * this->v + (t & 1u), t >> 1);
            }
        }
    }
};

// Passes of three or four row blocks (a slot holds four tiles): bound by the matrix
// cores and the loads' issue (900 cycles of MFMA per SIMD and row block for a step's
// 32 KB of weights and 10 KB of rows per block). A step is 128 columns.
template <bool UP, uint32_t NB>
struct QWide : QBase<UP, NB, 1> {
    using QB = QBase<UP, NB, 1>;
    using QB::P;
    struct WB {
        u32x4 w[4];
        uint32_t s[2];
    };
    static constexpr uint32_t kLoads = 5;
    f32x4 acc[4][NB];

    WL_MEM QWide(const DecodeArgs& a_, const BatchArgs& b_) : QB{a_, b_} {}
    WL_MEM void load(uint32_t s, WB& W, uint32_t j) const {
        const rsrc_t rs = make_rsrc(this->wbase, this->wbytes);
        if (j < 4u) {
            uint32_t ch;  // UP: slice j; down: slice 2s + (j & 1) of row pair j / 2
            if (UP) ch = min(this->wpart * 4u + j, this->S - 1u) * 8u * this->nk + s;
            else ch = (2u * s + j % 2u) * this->nq + min(16u * this->wpart + 2u * this->v + j / 2u, this->nq - 1u);
            W.w[j] = bld16(rs, this->vw, ch * 1024u);
        } else {
            const uint32_t so = (this->wpart * 8u * this->nst2 + s / 2u) * 512u;
            if (UP) bld8(rs, this->vs, so, W.s);
            else W.s[0] = __builtin_amdgcn_raw_buffer_load_b32(rs, (int)this->vs, (int)(so + 4u * (s & 1u)), 0);
        }
    }
    WL_MEM void begin(uint32_t i) {
        this->begin_unit(i);
#pragma unroll
        for (uint32_t t = 0; t < 4; t++)
#pragma unroll
            for (uint32_t m = 0; m < NB; m++) acc[t][m] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    template <class Next>
    WL_MEM void comp(uint32_t s, const uint8_t* sl, WB& W, Next next) {
        constexpr uint32_t N = P * NB, AH = 2u;
        i32x8 af[AH + 1u];
        u32x2 sa[NB];
        const uint32_t lo16 = this->lo16;
        auto frag = [&](uint32_t it) { return q_frag(sl + (it % NB) * QB::kTileB, it / NB, lo16, this->lo8); };
#pragma unroll
        for (uint32_t it = 0; it < AH; it++) af[it] = frag(it);
#pragma unroll
        for (uint32_t m = 0; m < NB; m++) sa[m] = q_scales(sl + m * QB::kTileB, this->lo8);
        // the step's scale bytes: UP the step's k tile of the word's two (byte 2
        // (i & 1)), down as the weights' halves (byte h)
        if (UP) {
            W.s[0] >>= 8u * (s & 1u);
            W.s[1] >>= 8u * (s & 1u);
        } else {
            uint32_t lo, hi;
            swap32(W.s[0], W.s[0] >> 16, lo, hi);
            W.s[0] = lo;
            W.s[1] = hi;
            pair_swap(W.w[0], W.w[1]);
            pair_swap(W.w[2], W.w[3]);
        }
#pragma unroll
        for (uint32_t it = 0; it < N; it++) {
            const uint32_t m = it % NB, p = it / NB;
            if (it + AH < N) af[(it + AH) % (AH + 1u)] = frag(it + AH);
            next(it, N);
#pragma unroll
            for (uint32_t t = 0; t < 4; t++) {
                // UP: slice t; down: row pair t / 2, half t % 2
                const uint32_t ow = UP ? 2u * (t & 1u) : t >> 1;
                const uint32_t sw = UP ? W.s[t >> 1] : W.s[t & 1u];
                acc[t][m] = mmq(W.w[t], af[it % (AH + 1u)], acc[t][m], ow, sw, p & 3u, p < 4u ? sa[m].x : sa[m].y);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    WL_MEM void finish() {
#pragma unroll
        for (uint32_t m = 0; m < NB; m++) {
            if constexpr (UP) {
                this->put_up(m, [&](uint32_t t) { return acc[t][m]; });
            } else {
#pragma unroll
                for (uint32_t t = 0; t < 4; t++) this->put_down(acc[t][m], m, 16u * this->cu.part + 2u * this->v + (t >> 1), t & 1u);
            }
        }
    }
};

// Calls of at most kGroupMax entries that run all phases (BatchArgs::group): the
// work-groups of bup_kernel find the experts' counts, offsets and entries from the
// ids by themselves, and the first also stores them for the kernels after it. bcount
// and bscatter, a launch of 5 us each, take all other calls. An expert is chosen at
// most once per token, so a bit per token and expert gives counts and ranks
// (comparing every entry with all before it took 9 us at 64 tokens of 8 experts, all
// of it before the first load of a weight).
constexpr uint32_t kGroupMax = 4u * kGT;
// Words of token bits of an expert; they have to fit a slot.
__host__ __device__ inline uint32_t group_words(uint32_t T) { return (T + 31u) / 32u; }
// Afterwards ent[r] is the token of compact entry r (in the place of the token table).
// (id: this thread's entries' experts, entry threadIdx.x + kGT r in id[r].)
WL_DEV void group_entries(const BatchArgs& b, uint32_t E, uint32_t K, const ExpertTab& et, uint16_t* ent,
                          const uint32_t (&id)[kGroupMax / kGT]) {
    constexpr uint32_t N = kGroupMax / kGT;
    const uint32_t n = b.T * K, i = threadIdx.x, lane = i & 63u, nw = group_words(b.T);
    uint32_t* bits = (uint32_t*)slot<0>();  // (free until the first pipeline)
    uint32_t t[N], rank[N];
#pragma unroll
    for (uint32_t r = 0; r < N; r++) t[r] = (i + r * kGT) / K;
    for (uint32_t f = i; f < E * nw; f += kGT) bits[f] = 0u;
    lds_barrier();
#pragma unroll
    for (uint32_t r = 0; r < N; r++)
        if (i + r * kGT < n) atomicOr(bits + id[r] * nw + t[r] / 32u, 1u << (t[r] % 32u));
    lds_barrier();
    for (uint32_t f = i; f < E; f += kGT) {
        uint32_t c = 0;
        for (uint32_t w = 0; w < nw; w++) c += (uint32_t)__popc(bits[f * nw + w]);
        et.cnt[f] = c;
    }
#pragma unroll
    for (uint32_t r = 0; r < N; r++) {
        rank[r] = 0u;
        if (i + r * kGT >= n) continue;
        for (uint32_t w = 0; w < t[r] / 32u; w++) rank[r] += (uint32_t)__popc(bits[id[r] * nw + w]);
        rank[r] += (uint32_t)__popc(bits[id[r] * nw + t[r] / 32u] & ((1u << (t[r] % 32u)) - 1u));
    }
    lds_barrier();
    if (i < 64u) {
        const uint32_t per = cdiv(E, 64u), e0 = lane * per;
        uint32_t mine = 0;
        for (uint32_t f = e0; f < min(e0 + per, E); f++) mine += et.cnt[f];
        uint32_t inc = mine;
#pragma unroll
        for (uint32_t o = 1; o < 64u; o <<= 1) {
            const uint32_t t0 = __shfl_up(inc, o, 64);
            if (lane >= o) inc += t0;
        }
        uint32_t off = inc - mine;
        for (uint32_t f = e0; f < min(e0 + per, E); f++) {
            et.off[f] = off;
            off += et.cnt[f];
        }
    }
    lds_barrier();
    const bool put = blockIdx.x == 0u;
#pragma unroll
    for (uint32_t r = 0; r < N; r++) {
        const uint32_t en = i + r * kGT;
        if (en >= n) continue;
        const uint32_t c = et.off[id[r]] + rank[r];
        ent[c] = (uint16_t)t[r];
        if (put) {
            gst(b.ent + c, en);
            gst(b.pos + en, c);
        }
    }
    if (!put) return;
    for (uint32_t f = i; f < E; f += kGT) {
        gst(b.counts + f, et.cnt[f]);
        gst(b.offsets + f, et.off[f]);
    }
    if (i == 0u) gst(b.offsets + E, n);
}
template <bool UP>
WL_DEV ExpertTab load_expert_tab(const BatchArgs& b, uint32_t E, uint32_t K, uint32_t* s, const uint8_t* const* stab,
                                 const uint32_t (&ids)[kGroupMax / kGT]) {
    const ExpertTab et{s, s + E, s + 2u * E, s + 3u * E + 1u, s + 3u * E + 1u + kGW};
    const bool skip = (b.flags & kBatchSkipUnbound) != 0u;
    const uint32_t esh = (b.flags & kBatchShared4) ? E - 1u : E;
    const bool group = UP && b.group != 0u;
    if (group) group_entries(b, esh, K, et, (uint16_t*)(dyn_lds() + tok_table_offset(esh)), ids);
    uint32_t sizes = 0, sums = 0;
    for (uint32_t f = threadIdx.x; f < E; f += kGT) {
        uint32_t c;
        bool here = true;  // its passes are this launch's
        if (f == esh) {
            c = b.T;
            here = !(b.flags & kBatchNoShared);
            et.off[f] = b.T * K;
        } else if (group) {
            c = et.cnt[f];
        } else {
            // stab[f] was written by this thread (load_slot_tab, same stride)
            c = gld(b.counts + f);
            here = !skip || stab[f] != nullptr;
            et.off[f] = gld(b.offsets + f);
        }
        et.cnt[f] = here ? c : 0u;
        const PassSplit sp = pass_split(c, false);
        if (here) sizes |= sp.sizes();
        sums += sp.np + ((cdiv(c, kRB) - sp.np) << 16);
    }
#pragma unroll
    for (uint32_t o = 1; o < 64u; o <<= 1) {
        sizes |= __shfl_xor(sizes, (int)o, 64);
        sums += __shfl_xor(sums, (int)o, 64);
    }
    if ((threadIdx.x & 63u) == 0u) {
        et.sizes[threadIdx.x >> 6] = sizes;
        et.sums[threadIdx.x >> 6] = sums;
    }
    return et;
}
// The routed passes of NB row blocks at pl; returns their units' count.
template <bool UP, uint32_t NB, bool FOLD = false>
WL_DEV uint32_t run_routed(const DecodeArgs& a, const BatchArgs& b, uint32_t E, const ExpertTab& et,
                           const uint8_t* const* stab, Places pl, bool any, bool single) {
    using Kn = std::conditional_t<(NB > 2u), QWide<UP, NB>, QNarrow<UP, NB, FOLD>>;
    const PassTab pt = load_pass_tab(et, E, NB, single);
    pipeline_drain();
    const uint32_t H = a.H, I = a.I;
    Kn w(a, b);
    w.H = H;
    w.I = I;
    w.E = E;
    w.K = a.K;
    w.nk = (UP ? H : I) / 128u;
    w.S = I / kSlice;
    w.nq = H / 32u;
    w.parts = UP ? cdiv(w.S, 4u) : cdiv(w.nq, 16u);
    w.nst2 = cdiv(UP ? H : I, 256u);
    w.nst = NB > 2u ? w.nk : w.nst2;
    const uint32_t U = pt.n * w.parts, end = pl.base + U, G = gridDim.x;
    w.any = any;
    w.pl = pl;
    // gate/up of one row block: the units of the last round, where at most half of
    // the work-groups have one, go to two or four of them each (not with a token table:
    // it is sized for cdiv(U, G) units of a work-group)
    w.tail = end;
    w.cut = 0u;
    if (UP && NB == 1u && b.group && end > G) {
        const uint32_t rem = (end - G) % G;
        w.cut = rem == 0u || rem > U || 2u * rem > G ? 0u : 4u * rem > G ? 1u : 2u;
        if (w.cut) w.tail = end - rem;
    }
    w.nu = pl.count(w.tail + ((end - w.tail) << w.cut));
    w.lane = threadIdx.x & 63u;
    w.v = uni(threadIdx.x >> 6);
    w.lo8 = q_lo8();
    w.lo16 = q_lo16();
    w.pt = pt;
    w.stab = stab;
    w.NL = NativeLayout::make(H, I);
    w.vw = (UP ? (uint32_t)w.NL.gu + w.v * w.nk * 1024u : (uint32_t)w.NL.dn) + 16u * w.lane;
    w.vs = (uint32_t)(UP ? w.NL.bgus : w.NL.bdns) + w.v * w.nst2 * 512u + 8u * w.lane;
    if (UP) {
        uint16_t* tt = (uint16_t*)(dyn_lds() + tok_table_offset(a.E));
        w.tt = tt;
        if (!b.group) fill_tokens(w, tt, kRB * NB);
    }
    run_units(w);
    return U;
}
// The layer's units: the shared expert's, then the routed passes from the largest.
// Routed rows as fp6 pieces against fp4 weights run at 3.5 times the rate of bf16
// pieces and need no conversion of the weights. Whole calls, hidden 6144, inter
// 2048, 8 of 256 experts (256 work-groups of eight waves), before (bf16 pieces,
// passes of 32 and 64) and now: 4096 tokens 8435 and 5165 us, 1000 tokens 2309 and
// 1594, 64 tokens (one row block per expert; the weights' 4.4 GB at 6.2 TB/s) 735 and
// 732, 7 tokens 209 and 205; hidden 2944, inter 1408, 6 of 160 experts, 333 tokens: 465 and 313.
// Error against 64 bits: 8.1e-7 and 4.6e-7 at 4096 tokens, 3.6e-7 and 1.5e-7 at 64.
template <bool UP>
WL_DEV void run_gemm(const DecodeArgs* pa, const BatchArgs& b) {
    const DecodeArgs& a = *pa;
    uint8_t* dyn = dyn_lds();
    const bool sh4 = (b.flags & kBatchShared4) != 0u;
    // (the loads of the tables go out together, as their waits are the head of the
    // kernel)
    const uint32_t more = gld(b.more + (UP ? 0 : 1));
    uint32_t ids[kGroupMax / kGT];
    if (UP && b.group) {
#pragma unroll
        for (uint32_t r = 0; r < kGroupMax / kGT; r++)
            ids[r] = (uint32_t)gld(b.idx + min(threadIdx.x + r * kGT, b.T * a.K - 1u));
    }
    const uint32_t E = a.E + (sh4 ? 1u : 0u);  // experts in the pass table
    const uint8_t* const* stab = load_slot_tab(a, a.E, sh4, (const uint8_t**)dyn);
    const ExpertTab et = load_expert_tab<UP>(b, E, a.K, (uint32_t*)(dyn + 8u * E), stab, ids);
    uint32_t u = run_shared_expert<UP>(a, b);
    // (a pass over more than 32 tokens takes one and a half to two times a routed unit:
    // 80 tokens 804 to 791 us, 96 841 to 828; past 128 there are too many)
    const uint32_t skip = b.T > 32u && b.T <= 128u && u < gridDim.x && (!UP || b.group) ? u : 0u;
    // (pass sizes that no expert has cost a table of 2 us each where they were
    // looked up one by one)
    lds_barrier();
    uint32_t sizes = 0, sums = 0;
#pragma unroll
    for (uint32_t w = 0; w < kGW; w++) {
        sizes |= et.sizes[w];
        sums += et.sums[w];
    }
    sizes = uni(sizes);
    sums = uni(sums);
    // Few larger passes among many small ones run as passes of one block, if that adds
    // at most a 64th to the weights read: a pipeline of their own, a unit or two for
    // some of the work-groups, had these end last (at 64 tokens, one expert of two
    // blocks among 213: by 17 us of 465, bdown 28 of 271). All experts of the call
    // count, so that one whose experts come in groups gives the same bits.
    const bool single = sums >> 16 != 0u && 64u * (sums >> 16) <= (sums & 0xFFFFu);
    if (single && sizes) sizes = 2u;
    const bool any = uni(more) != 0u;
    if (sizes & 1u << 4) u += run_routed<UP, 4>(a, b, E, et, stab, Places::from(u, skip), any, single);
    if (sizes & 1u << 3) u += run_routed<UP, 3>(a, b, E, et, stab, Places::from(u, skip), any, single);
    if (sizes & 1u << 2) u += run_routed<UP, 2>(a, b, E, et, stab, Places::from(u, skip), any, single);
    if (sizes & 1u << 1) {
        if (any) run_routed<UP, 1, true>(a, b, E, et, stab, Places::from(u, skip), any, single);
        else run_routed<UP, 1>(a, b, E, et, stab, Places::from(u, skip), any, single);
    }
}
