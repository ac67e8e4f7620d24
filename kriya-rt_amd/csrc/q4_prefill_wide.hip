// q4_prefill_wide.hip — prefill Q4_G64 matmul with wide wave tiles on v_mfma_f32_32x32x16_f16.
//
// The same operation, operands and epilogues as q4_prefill.hip (launch_rules.hpp says which of the two a launch
// takes; odd 64-group counts stay there); replaces the reference's M >= 64 simdgroup kernels
// (kernels/metal/q4_gemm_and_moe.metal:2708-3215) where there are enough tiles to fill the chip.
//
// What bounds it: instruction issue beside the matrix cores, and at large M the power limit.  A register
// micro-benchmark of this inner loop (dequantisation and LDS reads included) holds 2350 TFLOP/s on constant
// data and 1480 on random data, where the clock drops.  So the design keeps the instructions per matrix
// instruction low:
//   * 32x32x16 matrix instructions: 32 cycles each, so about six other instructions issue under one (with
//     16x16x32 three VALU per MFMA already cost 28 % in the same micro-benchmark);
//   * a wave owns MF x 32 token rows by NF x 32 weight rows and dequantises its own weight rows into the A
//     operand: 13 VALU per 8 weights, shared by MF matrix instructions (one shift per word: the odd nibbles
//     come out as 16 q and are scaled by an exact fp16 fma);
//   * the next fragment's dequantisation, the LDS reads of the next slice and the next step's requests are
//     issued piecewise between the matrix instructions (pinned by scheduling barriers): requests issued
//     together hold a wave for about 45 cycles each;
//   * scales and biases come in one 8-byte load per row and four steps (lane half h holds steps 2 h and
//     2 h + 1) and reach the lanes by ds_bpermute;
//   * the epilogue passes 32 token rows at a time through a wave-private LDS tile (no block barriers; four
//     consecutive columns per LDS write, eight per global store), and is kept short: unrolled tanh and
//     per-element tails made it 11 us per block through the instruction cache, 5 us now.
// Measured (K = 2048, 11008 gate/up pairs, m = 3907): 482 us on the 16x16x32 kernel, 327 here (373 in the first ten
// launches after idle, before the clock has settled); the down projection 2048 x 11008, 413 -> 174 us; [12288, 4096] at
// m = 512 / 2048 88 / 425 -> 65 / 196 us.  Counters of these two launches: matrix cores busy 62 % and 50 % of SIMD cycles,
// 5.6 and 4.7 VALU per matrix instruction (gate/up with the epilogue's), waves waiting to issue (SQ_WAIT_INST_ANY) 44 and
// 26 % of their cycles and for memory or barriers (SQ_WAIT_ANY) 19 and 28 %, LDS bank conflicts 4 and 1 %.
//
// Column order: lane (c, h) of a 128-column step holds the 64 columns of group 2 g + h of weight row c (two
// 16-byte loads); slice j multiplies word j of both halves, i.e. columns 64 h + 8 j .. + 7, so X is read
// from LDS at unit 8 h + j.  Inside a unit the order is the nibble-pair order of the dequantiser.
#include <type_traits>

#include "kr_internal.hpp"
#include "launch_rules.hpp"
#include "q4_prefill.hpp"

namespace kr {

namespace {

// Those of src[0 .. 7] (outputs n .. n + 7 of x) that are not finite, again in plain f32 over columns c0 .. c1 - 1.  All
// eight at a time: their loads overlap.  Only these outputs: one row of 1e5 in 512, [12288, 4096], takes 1.15 ms (whole
// tiles: 26.7, 11.8 with the 64 x 64 tiles of q4_prefill.hip).
__device__ __forceinline__ void exact8(const Q4Mat &w, uint32_t n, const uint16_t *x, uint32_t K, uint32_t c0, uint32_t c1,
                                       float *src) {
    bool any = false;
#pragma unroll
    for (int e = 0; e < 8; ++e) any |= !__builtin_isfinite(src[e]);
    if (!any) return;
    float sum[8] = {};
#pragma unroll 1
    for (uint32_t c = c0; c < c1; c += 8) {
        const u32x4 v = *reinterpret_cast<const u32x4 *>(x + c);
        const uint32_t X[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const size_t row = min(n + e, w.n - 1);
            const uint32_t q = w.qw[row * (K >> 3) + (c >> 3)];
            const float s = bf16_to_f32(w.sc[row * (K >> 6) + (c >> 6)]), b = bf16_to_f32(w.bi[row * (K >> 6) + (c >> 6)]);
#pragma unroll
            for (int j = 0; j < 8; ++j)
                sum[e] = fmaf(fmaf((float)((q >> (4 * j)) & 15u), s, b),
                              __uint_as_float(j & 1 ? X[j >> 1] & 0xFFFF0000u : X[j >> 1] << 16), sum[e]);
        }
    }
#pragma unroll
    for (int e = 0; e < 8; ++e)
        if (!__builtin_isfinite(src[e])) src[e] = sum[e];
}

// 16-byte epilogue accesses: the launch's outputs (or partials) and bias allow them.
template <int EPI>
__device__ __forceinline__ bool prefill_vec_out(const MfmaArgs &args, const MfmaProblem &P) {
    if (EPI == kMfmaPartial) return (uintptr_t)args.partial % 16 == 0 && P.w.n % 8 == 0;
    return (uintptr_t)P.out % 16 == 0 && P.ldo % 8 == 0 && (!P.bias || (uintptr_t)P.bias % 16 == 0);
}

// Eight consecutive output columns n .. n + 7 of token row m from LDS (src, 16-byte aligned, the activation
// applied): bias, accumulation and the store, in 16-byte pieces when `vec`.  Columns beyond N are dropped.
template <int EPI, bool kGateUp>
__device__ __forceinline__ void prefill_store8(const MfmaArgs &args, const MfmaProblem &P, uint32_t ks, uint32_t m,
                                               uint32_t n, float *src, bool vec) {
    const uint32_t N = P.w.n;
    const bool full = vec && n + 8 <= N;
    if (kGateUp && args.act != 0) {  // rolled: the tanh of eight columns is long code
#pragma unroll 1
        for (int e = 0; e < 8; ++e) src[e] = activation(src[e], args.act) * src[32 + e];
    }
    f32x4 lo = reinterpret_cast<const f32x4 *>(src)[0], hi = reinterpret_cast<const f32x4 *>(src)[1];
    if (kGateUp && args.act == 0) {
        const f32x4 ul = reinterpret_cast<const f32x4 *>(src)[8], uh = reinterpret_cast<const f32x4 *>(src)[9];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            lo[e] = activation(lo[e], 0) * ul[e];
            hi[e] = activation(hi[e], 0) * uh[e];
        }
        if (!full) {
            reinterpret_cast<f32x4 *>(src)[0] = lo;
            reinterpret_cast<f32x4 *>(src)[1] = hi;
        }
    }
    if constexpr (EPI == kMfmaPartial) {
        static_assert(!kGateUp, "partials of one matrix");
        float *dst = args.partial + ((size_t)ks * args.m + m) * (size_t)N + n;
        if (full) {
            reinterpret_cast<f32x4 *>(dst)[0] = lo;
            reinterpret_cast<f32x4 *>(dst)[1] = hi;
        } else {
#pragma unroll 1
            for (uint32_t e = 0; e < 8 && n + e < N; ++e) dst[e] = src[e];
        }
        return;
    }
    const size_t o = (size_t)m * P.ldo + n;
    if (full) {
        auto add_bf16 = [&](u32x4 b) {
            const uint32_t bb[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                f32x4 &t = e < 2 ? lo : hi;
                t[2 * (e & 1)] += bf16_to_f32(bb[e] & 0xFFFFu);
                t[2 * (e & 1) + 1] += bf16_to_f32(bb[e] >> 16);
            }
        };
        if (P.bias) add_bf16(*reinterpret_cast<const u32x4 *>(P.bias + n));
        if (args.out_f32) {
            f32x4 *out = reinterpret_cast<f32x4 *>(reinterpret_cast<float *>(P.out) + o);
            if (args.accumulate) {
                lo += out[0];
                hi += out[1];
            }
            out[0] = lo;
            out[1] = hi;
        } else {
            u32x4 *out = reinterpret_cast<u32x4 *>(reinterpret_cast<uint16_t *>(P.out) + o);
            if (args.accumulate) add_bf16(out[0]);
            const u32x4 pk = {pack_bf16_rne(lo[0], lo[1]), pack_bf16_rne(lo[2], lo[3]), pack_bf16_rne(hi[0], hi[1]),
                              pack_bf16_rne(hi[2], hi[3])};
            out[0] = pk;
            if (kGateUp && args.out_h)  // the same 8 values as the next projection's fp16 operand
                *reinterpret_cast<u32x4 *>(args.out_h + o) = x_unit_f16(pk);
        }
        return;
    }
    // column by column from the LDS tile (a run-time index into registers would be moves), rolled: tails only
#pragma unroll 1
    for (uint32_t e = 0; e < 8 && n + e < N; ++e) {
        float x = src[e];
        if (P.bias) x += bf16_to_f32(P.bias[n + e]);
        if (args.out_f32) {
            float *out = reinterpret_cast<float *>(P.out);
            out[o + e] = args.accumulate ? out[o + e] + x : x;
        } else {
            uint16_t *out = reinterpret_cast<uint16_t *>(P.out);
            const uint32_t b = f32_to_bf16(args.accumulate ? x + bf16_to_f32(out[o + e]) : x);
            out[o + e] = (uint16_t)b;
            if (kGateUp && args.out_h) {  // element e of its 8-column unit goes to 2 (e % 4) + e / 4
                const _Float16 hv = (_Float16)bf16_to_f32(b);
                const uint32_t c = n + e;
                args.out_h[o - n + (c & ~7u) + 2 * (c & 3u) + ((c & 7u) >> 2)] = __builtin_bit_cast(uint16_t, hv);
            }
        }
    }
}

// MF x 32 token rows by 4 waves x NF x 32 weight rows per block.
template <int MF, int NF, int NW>
struct WideTile {
    static constexpr int kBM = MF * 32;
    static constexpr int kCols = 4 * NF * 32 / NW;   // output columns per block
    static constexpr int kBuf = kBM * 256;           // one 128-column X slice in fp16
    static constexpr int kTile = 4 * 32 * (NF * 32 + 4) * 4;  // the epilogue's LDS tiles
    static constexpr int kLds = 2 * kBuf > kTile ? 2 * kBuf : kTile;
};

template <int MF, int NF, int NW, bool CVT, int EPI, int OCC>
__global__ __launch_bounds__(256, OCC) void q4_prefill_wide_kernel(MfmaArgs args) {
    using T = WideTile<MF, NF, NW>;
    extern __shared__ __align__(16) char lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 31, h = lane >> 5;

    // ---- block -> (K split, problem, m tile, n tile).  Workgroups go to the 8 XCDs (each with its own L2)
    // round-robin in launch order: XCD j takes the j-th contiguous part of the tiles (with a split K: of all
    // splits' tiles, split by split, so that an L2 holds one K range of X; args.xcd_tiles == 0: of each
    // split's tiles).  Within a problem groups of 8 m tiles run through the n tiles, so that the tiles an
    // XCD works on at a time share X rows and weight rows.  Any grid maps one-to-one.
    const uint32_t nblk = gridDim.x;
    const uint32_t total = args.xcd_tiles ? nblk * gridDim.y : nblk;
    uint32_t L = args.xcd_tiles ? blockIdx.x + blockIdx.y * nblk : blockIdx.x;
    {
        const uint32_t j = L & 7, q = total >> 3, r = total & 7;
        L = j * q + min(j, r) + (L >> 3);
    }
    const uint32_t ks = args.xcd_tiles ? L / nblk : blockIdx.y, bid = L % nblk;
    int pi = 0;
#pragma unroll
    for (int i = 1; i < kMaxMfmaProblems; ++i)
        if (i < args.np && bid >= args.p[i].tile_begin) pi = i;
    const MfmaProblem &P = args.p[pi];
    const uint32_t N = P.w.n, M = args.m, K = args.k, G = K >> 6, GS = K >> 7;
    const uint32_t tiles_m = (M + T::kBM - 1) / T::kBM, tiles_n = (N + T::kCols - 1) / T::kCols;
    uint32_t mt, nt;
    {
        constexpr uint32_t kGroupM = 8;
        const uint32_t local = bid - P.tile_begin, per = kGroupM * tiles_n;
        const uint32_t grp = local / per, in = local % per, gm = min(tiles_m - grp * kGroupM, kGroupM);
        mt = grp * kGroupM + in % gm;
        nt = in / gm;
    }
    const uint32_t m0 = mt * T::kBM;
    const uint32_t g_begin = ks * (args.groups_per_split / 2), g_end = min(GS, g_begin + args.groups_per_split / 2);
    const uint32_t nsteps = g_end > g_begin ? g_end - g_begin : 0;

    const uint32_t kMask0 = opaque_s(0x000F000Fu), kMask1 = opaque_s(0x00F000F0u);
    const uint32_t kMagic = opaque_v(0x64006400u);

    const uint32_t rowbytes = K >> 1;
    rsrc_t rq[2], rs[2], rb[2];
#pragma unroll
    for (int i = 0; i < NW; ++i) {
        const bool second = NW == 2 && (i & 1);
        const Q4Mat &w = second ? P.w2 : P.w;
        rq[i] = make_rsrc(w.qw, N * rowbytes);
        rs[i] = make_rsrc(w.sc, N * G * 2);
        rb[i] = make_rsrc(w.bi, N * G * 2);
    }
    uint32_t oq[NF], os[NF];
#pragma unroll
    for (int f = 0; f < NF; ++f) {
        const uint32_t F = wave * NF + f;  // gate/up: fragments alternate gate, up of the same rows
        const uint32_t row = min(nt * T::kCols + (NW == 2 ? F >> 1 : F) * 32 + c, N - 1);  // tail rows never stored
        oq[f] = row * rowbytes + h * 32;
        os[f] = row * G * 2 + h * 8;
    }
    // X staging as in q4_prefill.hip: row r, unit u in slot r * 16 + (u ^ swizzle(r)), by direct-to-LDS loads
    auto swizzle = [](uint32_t r) -> uint32_t { return ((r & 7) << 1) | ((r >> 3) & 1); };
    constexpr int XI = T::kBM * 16 / 64 / 4;
    const rsrc_t rx = make_rsrc(CVT ? args.x : args.xh, (M - 1) * args.ldx * 2 + K * 2);
    uint32_t xo[XI];
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        const uint32_t r = (wave * XI + i) * 4 + (lane >> 4), u = (uint32_t)(lane & 15) ^ swizzle(r);
        xo[i] = min(m0 + r, M - 1) * args.ldx * 2 + u * 16;
    }
    auto dma_x = [&](uint32_t g, int buf, int i) {
        dma16(rx, lds + buf * T::kBuf + (wave * XI + i) * 1024, xo[i], g * 256);
    };
    // the lane's own 16 bytes of DMA instruction i, converted where they landed
    auto x_slot = [&](int buf, int i) {
        return reinterpret_cast<u32x4 *>(lds + buf * T::kBuf + (wave * XI + i) * 1024 + lane * 16);
    };
    // slice j of a step: unit 8 h + j of rows 32 a + c
    const uint32_t xa0 = c * 256 + (((8u * h) ^ swizzle(c)) << 4);

    u32x4 w[2][NF][2];
    u32x2 sreg[NF], breg[NF];
    auto load_q = [&](uint32_t g, u32x4(&r)[NF][2], int f, int q) {
        r[f][q] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rq[f & (NW - 1)], oq[f] + q * 16, g * 64, 0));
    };
    // the scale and bias pairs of four steps: lane half h holds those of steps 2 h, 2 h + 1
    auto load_sb = [&](uint32_t g) {
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            sreg[f] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs[f & (NW - 1)], os[f], g * 4, 0));
            breg[f] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rb[f & (NW - 1)], os[f], g * 4, 0));
        }
    };
    const uint32_t hsel = h ? 0x07060c0cu : 0x05040c0cu;

    f32x16 acc[MF][NF];
#pragma unroll
    for (int a = 0; a < MF; ++a)
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[a][f][v] = 0.0f;

    const f16x2_t k1024 = {(_Float16)-1024.0f, (_Float16)-1024.0f};
    const f16x2_t k16 = {(_Float16)0.0625f, (_Float16)0.0625f}, k64 = {(_Float16)-64.0f, (_Float16)-64.0f};
    // One word's dequantisation in four pieces, issued one after each matrix instruction.
    struct Dq {
        uint32_t q, q8, t0, t1, t2, t3;
        f16x2_t h0, h1, h2, h3, p0, p1, p2, p3;
    };
    auto dq_piece = [&](auto A, Dq &d, f16x2_t s2, f16x2_t b2) {
        constexpr int a = decltype(A)::value;
        if constexpr (a == 0) {
            d.t0 = (d.q & kMask0) | kMagic;
            d.t1 = (d.q & kMask1) | kMagic;
            d.q8 = d.q >> 8;
            d.h0 = __builtin_bit_cast(f16x2_t, d.t0) + k1024;
        } else if constexpr (a == 1) {
            d.h1 = __builtin_elementwise_fma(__builtin_bit_cast(f16x2_t, d.t1), k16, k64);
            d.t2 = (d.q8 & kMask0) | kMagic;
            d.t3 = (d.q8 & kMask1) | kMagic;
            d.p0 = __builtin_elementwise_fma(d.h0, s2, b2);
        } else if constexpr (a == 2) {
            d.h2 = __builtin_bit_cast(f16x2_t, d.t2) + k1024;
            d.p1 = __builtin_elementwise_fma(d.h1, s2, b2);
            d.h3 = __builtin_elementwise_fma(__builtin_bit_cast(f16x2_t, d.t3), k16, k64);
        } else if constexpr (a == 3) {
            d.p2 = __builtin_elementwise_fma(d.h2, s2, b2);
            d.p3 = __builtin_elementwise_fma(d.h3, s2, b2);
        }
    };
    auto dq_frag = [](const Dq &d) {
        return f16x8_t{d.p0.x, d.p0.y, d.p1.x, d.p1.y, d.p2.x, d.p2.y, d.p3.x, d.p3.y};
    };
    constexpr int kPieces = MF >= 4 ? 1 : 4 / MF;  // dequantisation pieces per matrix instruction

    // scale and bias of step i (of this K group), of the lane's 64-column group, as fp16 pairs
    f16x2_t s2[2][NF], b2[2][NF];
    auto scales = [&](auto U, uint32_t i) {
        constexpr int u = decltype(U)::value;
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            const uint32_t sv = __builtin_amdgcn_ds_bpermute(c * 4 + (i & 2) * 64, sreg[f][u]);
            const uint32_t bv = __builtin_amdgcn_ds_bpermute(c * 4 + (i & 2) * 64, breg[f][u]);
            const _Float16 sh = (_Float16)__uint_as_float(__builtin_amdgcn_perm(sv, 0u, hsel));
            const _Float16 bh = (_Float16)__uint_as_float(__builtin_amdgcn_perm(bv, 0u, hsel));
            s2[u][f] = f16x2_t{sh, sh};
            b2[u][f] = f16x2_t{bh, bh};
        }
    };

    // The 8 NF phases of a step: one weight fragment times MF row fragments each, with the next
    // fragment's dequantisation, the A reads kLook slices ahead and the next step's requests spread
    // over them (requests issued together at the step's start hold the wave about 45 cycles each).
    constexpr int kPhases = 8 * NF, kLook = MF >= 4 ? 1 : 2;
    constexpr int kWLoads = 2 * NF;
    // first phase of the X and of the weight requests; X converted in place in the last phases
    constexpr int kXPhases = CVT ? kPhases / 4 : kPhases / 2;
    constexpr int kXFirst = CVT ? 0 : kPhases / 4, kWFirst = CVT ? kPhases / 4 : 0;
    constexpr int kWPhases = kPhases / 4;
    auto step = [&](auto U, uint32_t i) {
        constexpr int u = decltype(U)::value;
        constexpr int b = u & 1;
        const uint32_t gn = min(g_begin + i + 1, GS - 1);
        const char *xb = lds + b * T::kBuf;
        f16x8_t af[kLook + 1][MF];
#pragma unroll
        for (int l = 0; l < kLook; ++l)
#pragma unroll
            for (int a = 0; a < MF; ++a) af[l][a] = *reinterpret_cast<const f16x8_t *>(xb + (xa0 ^ (l << 4)) + a * 8192);
        Dq d0;
        d0.q = w[b][0][0][0];
        static_for<4>([&](auto A) { dq_piece(A, d0, s2[u][0], b2[u][0]); });
        f16x8_t bc = dq_frag(d0);
        __builtin_amdgcn_sched_barrier(0);
        static_for<kPhases>([&](auto JF) {
            constexpr int p = JF, j = p / NF, f = p % NF;
            constexpr bool last = p + 1 == kPhases;
            constexpr int jn = last ? 0 : (p + 1) / NF, fn = last ? 0 : (p + 1) % NF;
            const uint32_t xn = xa0 ^ (((j + kLook) & 7) << 4);
            Dq d;
            d.q = w[b][fn][jn >> 2][jn & 3];
            static_for<MF>([&](auto A) {
                constexpr int a = A;
                acc[a][f] = __builtin_amdgcn_mfma_f32_32x32x16_f16(bc, af[j % (kLook + 1)][a], acc[a][f], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (f == 0 && j + kLook < 8)
                    af[(j + kLook) % (kLook + 1)][a] = *reinterpret_cast<const f16x8_t *>(xb + xn + a * 8192);
                if constexpr (!last)
                    static_for<kPieces>([&](auto Q) {
                        dq_piece(std::integral_constant<int, a * kPieces + Q>{}, d, s2[u][fn], b2[u][fn]);
                    });
                if constexpr (a == 0) {
                    if constexpr (p >= kXFirst && p < kXFirst + kXPhases) {
                        constexpr int k = p - kXFirst;
#pragma unroll
                        for (int q = XI * k / kXPhases; q < XI * (k + 1) / kXPhases; ++q) dma_x(gn, b ^ 1, q);
                    }
                    if constexpr (p >= kWFirst && p < kWFirst + kWPhases) {
                        constexpr int k = p - kWFirst;
#pragma unroll
                        for (int q = kWLoads * k / kWPhases; q < kWLoads * (k + 1) / kWPhases; ++q)
                            load_q(gn, w[b ^ 1], q >> 1, q & 1);
                    }
                }
                if constexpr (CVT && a == MF / 2 && p >= kPhases / 2) {
                    if constexpr (p == kPhases / 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kWLoads) : "memory");
                    constexpr int k = p - kPhases / 2;
#pragma unroll
                    for (int q = XI * k / (kPhases / 2); q < XI * (k + 1) / (kPhases / 2); ++q) {
                        u32x4 *x = x_slot(b ^ 1, q);
                        *x = x_unit_f16(*x);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            });
            if constexpr (!last) bc = dq_frag(d);
            if constexpr (p + 1 == kPhases / 2) {  // mid-step: the next step's scales
                scales(std::integral_constant<int, u ^ 1>{}, i + 1);
                __builtin_amdgcn_sched_barrier(0);
            }
        });
        if constexpr (!CVT) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the X slice has landed
        if constexpr (u == 0) {  // past the last use of the block's scales: the next four steps'
            if (i & 2) load_sb(min(g_begin + i + 2, GS - 1));
        }
        __syncthreads();
    };

    if (nsteps) {
#pragma unroll
        for (int q = 0; q < XI; ++q) dma_x(g_begin, 0, q);
        __builtin_amdgcn_sched_barrier(0);
        load_sb(g_begin);
#pragma unroll
        for (int q = 0; q < kWLoads; ++q) load_q(g_begin, w[0], q >> 1, q & 1);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * NF) : "memory");
        if constexpr (CVT) {
#pragma unroll
            for (int q = 0; q < XI; ++q) {
                u32x4 *x = x_slot(0, q);
                *x = x_unit_f16(*x);
            }
        }
        scales(std::integral_constant<int, 0>{}, 0);
        __syncthreads();
        uint32_t i = 0;
        for (; i + 2 <= nsteps; i += 2) {
            step(std::integral_constant<int, 0>{}, i);
            step(std::integral_constant<int, 1>{}, i + 1);
        }
        if (i < nsteps) step(std::integral_constant<int, 0>{}, i);
    }

    // A non-finite sum (an operand beyond fp16, or an infinite input: it never turns finite again) is computed again
    // below, in plain f32; 0 * acc is NaN where acc is not finite.
    float z[4] = {0, 0, 0, 0};
#pragma unroll
    for (int a = 0; a < MF; ++a)
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int v = 0; v < 16; ++v) z[v & 3] = fmaf(acc[a][f][v], 0.0f, z[v & 3]);
    const float zs = (z[0] + z[1]) + (z[2] + z[3]);
    const bool bad = __ballot(zs != zs) != 0ull;  // in this wave
    // every wave's direct-to-LDS loads have landed before a tile is written over the X buffers
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    // A lane holds, of token row c, the weight rows 8 q + 4 h + 0 .. 3 of each fragment: four consecutive
    // columns.  Each wave passes 32 rows at a time through its own LDS region (no block barriers) and
    // stores eight consecutive columns per lane.
    constexpr bool kPair = NW == 2 && NF == 2;             // the wave holds a gate fragment and its up fragment
    constexpr int kWCols = kPair ? 32 : NF * 32;           // columns a wave writes
    constexpr int kPitch = NF * 32 + 4;
    static_assert(NW == 1 || NF == 2, "gate/up waves hold whole pairs");
    float *tile = reinterpret_cast<float *>(lds) + wave * 32 * kPitch;
    const bool vec = prefill_vec_out<EPI>(args, P);
    const uint32_t n0 = nt * T::kCols + wave * kWCols;
#pragma unroll
    for (int p = 0; p < MF; ++p) {
#pragma unroll
        for (int f = 0; f < NF; ++f)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<f32x4 *>(tile + c * kPitch + f * 32 + 8 * q + 4 * h) =
                    f32x4{acc[p][f][4 * q], acc[p][f][4 * q + 1], acc[p][f][4 * q + 2], acc[p][f][4 * q + 3]};
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        constexpr int kUnits = kWCols / 8;
        if (bad) {
            const uint32_t c0 = g_begin * 128, c1 = min(g_end * 128, K);
#pragma unroll 1
            for (int it = 0; it < kUnits / 2; ++it) {
                const uint32_t r = (it * 64 + lane) / kUnits, cu = lane % kUnits;
                const uint32_t m = m0 + p * 32 + r, n = n0 + cu * 8;
                if (m >= M || n >= N) continue;
                const uint16_t *xr = args.x + (size_t)m * args.ldx;
                float *src = tile + r * kPitch + cu * 8;
                exact8(P.w, n, xr, K, c0, c1, src);
                if constexpr (kPair) exact8(P.w2, n, xr, K, c0, c1, src + 32);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
#pragma unroll 2
        for (int it = 0; it < kUnits / 2; ++it) {
            const uint32_t r = (it * 64 + lane) / kUnits, cu = lane % kUnits;
            const uint32_t m = m0 + p * 32 + r, n = n0 + cu * 8;
            if (m < M && n < N) prefill_store8<EPI, kPair>(args, P, ks, m, n, tile + r * kPitch + cu * 8, vec);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

template <int MF, int NF, int NW, bool CVT, int OCC>
hipError_t launch_wide_shape(MfmaArgs &a, hipStream_t s) {
    using T = WideTile<MF, NF, NW>;
    uint32_t tiles = 0;
    for (int i = 0; i < a.np; ++i) {
        a.p[i].tile_begin = tiles;
        tiles += ((a.m + T::kBM - 1) / T::kBM) * ((a.p[i].w.n + T::kCols - 1) / T::kCols);
    }
    if (a.ksplit <= 1) a.groups_per_split = a.k / 64;
    a.xcd_tiles = tuning().prefill_xcd_split ? 1 : 0;
    const dim3 grid(tiles, a.ksplit > 1 ? a.ksplit : 1);
    if (a.ksplit > 1) {
        if constexpr (NW == 1 && MF == 4 && NF == 2) {
            hipLaunchKernelGGL((q4_prefill_wide_kernel<MF, NF, NW, CVT, kMfmaPartial, OCC>), grid, dim3(256), T::kLds, s, a);
            const hipError_t e = hipGetLastError();
            return e != hipSuccess ? e : launch_splitk_reduce(a, NW, s);
        }
        return hipErrorInvalidValue;
    }
    hipLaunchKernelGGL((q4_prefill_wide_kernel<MF, NF, NW, CVT, kMfmaDirect, OCC>), grid, dim3(256), T::kLds, s, a);
    return hipGetLastError();
}

template <int MF, int NF, int OCC>
hipError_t launch_wide(MfmaArgs &a, hipStream_t s) {
    if constexpr (NF == 2) {
        if (a.p[0].w2.qw)
            return a.xh ? launch_wide_shape<MF, NF, 2, false, OCC>(a, s) : launch_wide_shape<MF, NF, 2, true, OCC>(a, s);
    }
    return a.xh ? launch_wide_shape<MF, NF, 1, false, OCC>(a, s) : launch_wide_shape<MF, NF, 1, true, OCC>(a, s);
}

}  // namespace

// Gate/up: 128 x 128 tiles (64 pairs) once they give 1.5 blocks per compute unit, else q4_prefill.hip's of the same
// size: in kr_q4_mlp (the whole call, us, this kernel / that one) [2 x 11008, 2048] at m = 512 (344 tiles) 103 / 100, 640
// (430) 115 / 125, 1024 164 / 177, 3907 503 / 845.  Plain projections: launch_rules.hpp.  (The same rule with and
// without converted operands: KR_OPT_PREFILL_OPERANDS must not change the bits.)
int prefill_wide_shape(const MfmaArgs &a) {
    if (tuning().prefill_kernel != 0 || a.k % 128 != 0 || a.ksplit > 1) return kPrefillNarrow;
    uint32_t ns[kMaxMfmaProblems];
    for (int i = 0; i < a.np; ++i) ns[i] = a.p[i].w.n;
    if (a.p[0].w2.qw)
        return prefill_tiles(a.m, ns, 1, 128, 128) * 4 >= 6 * (uint64_t)device_cus() ? kPrefillWide42 : kPrefillNarrow;
    return prefill_choice(a.m, ns, a.np, a.k, 1, false, (uint32_t)device_cus()).shape;
}

hipError_t launch_prefill_wide(MfmaArgs &a, int shape, hipStream_t s) {
    switch (shape) {
        case kPrefillWide42: return launch_wide<4, 2, 2>(a, s);
        case kPrefillWide22: return launch_wide_shape<2, 2, 1, true, 2>(a, s);
        case kPrefillWide21: return launch_wide_shape<2, 1, 1, true, 4>(a, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace kr
