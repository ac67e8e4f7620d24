// q4_grouped.hip — routed Q4_G64 experts as grouped matrix products on v_mfma_f32_32x32x16_bf16, for routings
// that give an expert more tokens than the few-token kernel (q4_skinny.hip) takes at a time.
// Replaces the reference's routed GEMV (kernels/metal/q4_gemm_and_moe.metal:2642-2698) at prefill sizes.
//
// Exactness.  As in the few-token kernel x stays bf16 and the weights stay exact: the products are x times the
// integers 128 + q (exact in bf16, summed in f32), and the affine map of every 64-column group is applied to
// the f32 results,  sum_c x_c (s q_c + b) = s D + b S - 128 s S,  D = sum_c x_c (128 + q_c),  S = sum_c x_c.
// The S terms are one more matrix instruction per 128 columns: S is split into three bf16 parts (24 bits: the
// f32 value), which meet b and -128 s (both exact in bf16).
//
// What bounds it: waiting.  At 1000 tokens x top 4 of 60 experts (hidden 2048, inter 1408) the counters of the gate/up
// launch have the matrix cores busy 23 % of SIMD cycles, 10 VALU per matrix instruction and the waves, two per SIMD,
// waiting 40 % of their cycles for memory and barriers (SQ_WAIT_ANY) and 30 % to issue (SQ_WAIT_INST_ANY; down: 21, 10,
// 42, 32); it reads 320 MB for 198 MB of weights and x, a weight row once per expert and 96 tokens.  Per 128 columns and
// 32 x 32 outputs a wave issues 9 matrix instructions (288 cycles), 32 FMAs, and 56 VALU of unpacking shared by the row
// fragments.  The few-token kernel's 16-row chunks unpack and sum across waves for every 16 tokens: 300 + 180 us there;
// here 121 + 63 us.
//
// Operands.  X rows come with the columns of every 8 in the order the nibble pairs unpack in
// (e0 e4 e1 e5 e2 e6 e3 e7) and one 16-byte unit (hi mid lo hi mid lo 0 0) of S per 64-column group:
// moe_x_prep_kernel writes both for x, the gate/up epilogue for its own output.  A block takes 128 weight rows
// (gate/up: 64 gate and the same 64 up rows) by up to 32 MF tokens of one expert; X and its S units go
// through LDS by direct-to-LDS loads, two steps of 128 columns deep; each wave unpacks its own 32 weight
// rows.  A block's row fragments beyond its tokens are not multiplied.
#include <algorithm>
#include <type_traits>

#include "kr_internal.hpp"
#include "launch_rules.hpp"
#include "q4_prefill.hpp"

namespace kr {

namespace {

typedef __bf16 bf16x2v __attribute__((ext_vector_type(2)));

// f32 S -> the 16-byte unit (hi mid | lo hi | mid lo | 0 0) of bf16 parts, S = hi + mid + lo
__device__ __forceinline__ u32x4 sum_unit(float s) {
    const uint32_t hi = pack_bf16_rne(s, 0.0f);
    const float r1 = s - __uint_as_float(hi << 16);
    const uint32_t mid = pack_bf16_rne(r1, 0.0f);
    const float r2 = r1 - __uint_as_float(mid << 16);
    const uint32_t lo = pack_bf16_rne(r2, 0.0f);
    return u32x4{hi | (mid << 16), lo | (hi << 16), mid | (lo << 16), 0u};
}

// 8 bf16 in element order -> the order e0 e4 e1 e5 e2 e6 e3 e7
__device__ __forceinline__ u32x4 pair_order(const u32x4 &v) {
    return u32x4{__builtin_amdgcn_perm(v.z, v.x, 0x05040100u), __builtin_amdgcn_perm(v.z, v.x, 0x07060302u),
                 __builtin_amdgcn_perm(v.w, v.y, 0x05040100u), __builtin_amdgcn_perm(v.w, v.y, 0x07060302u)};
}

// Sum of a unit's 8 values, then over the 8 lanes that hold a 64-column group; the same in all of them.
__device__ __forceinline__ float group_sum(const u32x4 &v) {
    const uint32_t X[4] = {v.x, v.y, v.z, v.w};
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) s += __uint_as_float(X[i] << 16) + __uint_as_float(X[i] & 0xFFFF0000u);
    s += __shfl_xor(s, 1);
    s += __shfl_xor(s, 2);
    s += __shfl_xor(s, 4);
    return s;
}

// One thread per 16-byte unit; k % 128 == 0, so a wave's 8-lane groups never straddle a row.
__global__ __launch_bounds__(256) void moe_x_prep_kernel(const u32x4 *x, u32x4 *xp, u32x4 *su, uint32_t units) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    const u32x4 v = x[min(i, units - 1)];
    const float s = group_sum(v);
    if (i >= units) return;
    xp[i] = pair_order(v);
    if ((i & 7) == 0) su[i >> 3] = sum_unit(s);
}

template <int MF>
struct GroupedTile {
    static constexpr int kBM = 32 * MF;
    static constexpr int kX = kBM * 256;             // X bytes of one 128-column step
    static constexpr int kBuf = kX + 4096;           // and its two S units per row (1 KB per wave's request)
    static constexpr int kPitch = 128 + 4;           // floats per row of the epilogue's tile
    static constexpr int kTile = 32 * kPitch * 4;
    static constexpr int kLds = 2 * kBuf > kTile ? 2 * kBuf : kTile;
};

template <int MF, bool kGateUp, int OCC>
__global__ __launch_bounds__(256, OCC) void q4_grouped_kernel(GroupedArgs a) {
    using T = GroupedTile<MF>;
    extern __shared__ __align__(16) char lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int c = lane & 31, h = lane >> 5;
    constexpr uint32_t kCols = kGateUp ? 64 : 128;  // output columns per block
    const uint32_t K = a.k, G = K >> 6, GS = K >> 7;
    const uint32_t ntiles = (a.rows + kCols - 1) / kCols;

    // ---- the block's expert and tiles.  Lane l covers experts l + 64 i; mtiles before each by a wave scan.
    uint32_t item = blockIdx.x, e = 0, base = 0, cnt = 0, mt = 0, nt = 0;
    {
        uint32_t lo[4], n[4], before[4], run = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t x = lane + 64u * i;
            lo[i] = x < a.experts ? a.offsets[x] : 0u;
            n[i] = x < a.experts ? a.offsets[x + 1] - lo[i] : 0u;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t t = (n[i] + T::kBM - 1) / T::kBM;
            uint32_t v = t;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const uint32_t o = __shfl_up(v, d);
                if (lane >= d) v += o;
            }
            before[i] = run + v - t;
            run += __builtin_amdgcn_readlane(v, 63);
        }
        const uint32_t total = run * ntiles;
        if (item >= total) return;
        // XCD j takes the j-th contiguous part of the items: an expert's tiles share an L2
        const uint32_t j = item & 7, q = total >> 3, r = total & 7;
        item = j * q + min(j, r) + (item >> 3);
        const uint32_t u = item / ntiles;  // expert by expert: all (n, m) tiles of an expert, m fastest
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t t = (n[i] + T::kBM - 1) / T::kBM;
            const uint64_t hit = __ballot(u >= before[i] && u < before[i] + t);
            if (hit) {
                const int src = __builtin_ctzll(hit);
                e = 64u * i + (uint32_t)src;
                base = __builtin_amdgcn_readlane(lo[i], src);
                cnt = __builtin_amdgcn_readlane(n[i], src);
                const uint32_t b4 = __builtin_amdgcn_readlane(before[i], src);
                const uint32_t te = (cnt + T::kBM - 1) / T::kBM, idx = item - b4 * ntiles;
                mt = idx % te;
                nt = idx / te;
            }
        }
    }
    const uint32_t p0 = base + mt * T::kBM;                    // first sorted position
    const uint32_t rows = min(cnt - mt * T::kBM, (uint32_t)T::kBM);
    const uint32_t na = (rows + 31) / 32;                      // row fragments with tokens

    // ---- weights: gate/up blocks have their gate rows in waves 0, 1 and the same up rows in waves 2, 3
    const bool second = kGateUp && wave >= 2;
    const Q4Mat &W = second ? a.w2 : a.w;
    const uint32_t rowbytes = K >> 1;
    // one expert's rows: offsets stay below 4 GiB whatever the number of experts
    const size_t er = (size_t)e * a.rows;
    const rsrc_t rq = make_rsrc(W.qw + er * (K >> 3), a.rows * rowbytes);
    const rsrc_t rs = make_rsrc(W.sc + er * G, a.rows * G * 2);
    const rsrc_t rb = make_rsrc(W.bi + er * G, a.rows * G * 2);
    const uint32_t wrow = min(nt * kCols + (kGateUp ? (wave & 1) : wave) * 32 + c, a.rows - 1);  // tail rows never stored
    const uint32_t oq = wrow * rowbytes + h * 16, os = wrow * G * 2 + h * 8;

    // ---- X rows: unit u of row r in slot r * 16 + (u ^ swizzle(r)); S units (two per row and step) after them
    auto swizzle = [](uint32_t r) -> uint32_t { return ((r & 7) << 1) | ((r >> 3) & 1); };
    auto x_row = [&](uint32_t r) -> uint32_t {  // row of X of the tile's row r (rows past the last repeat it)
        const uint32_t p = p0 + min(r, rows - 1);
        return a.x_div ? a.sorted[p] / a.x_div : p;
    };
    constexpr int XI = T::kBM * 16 / 256;  // X instructions per wave and step
    const rsrc_t rx = make_rsrc(a.xp, a.xrows * K * 2);
    const rsrc_t ru = make_rsrc(a.su, a.xrows * G * 16);
    uint32_t xo[XI];
#pragma unroll
    for (int i = 0; i < XI; ++i) {
        const uint32_t r = (i * 4 + wave) * 4 + (lane >> 4), u = (uint32_t)(lane & 15) ^ swizzle(r);
        xo[i] = x_row(r) * K * 2 + u * 16;
    }
    // S units: wave w loads those of rows 32 w + lane / 2 (waves past the tile repeat valid rows)
    const uint32_t uo = x_row(32 * min(wave, MF - 1) + (lane >> 1)) * G * 16 + (lane & 1) * 16;
    auto dma_x = [&](uint32_t g, int buf, int i) __attribute__((always_inline)) {
        dma16(rx, lds + buf * T::kBuf + (i * 4 + wave) * 1024, xo[i], g * 256);
    };
    auto dma_u = [&](uint32_t g, int buf) __attribute__((always_inline)) {
        dma16(ru, lds + buf * T::kBuf + T::kX + wave * 1024, uo, g * 32);
    };
    // slice j of group gr: unit 8 gr + 4 h + j of rows 32 a + c
    const uint32_t xa0 = c * 256 + (((4u * h) ^ swizzle(c)) << 4);
    const uint32_t ua = T::kX + c * 32 + h * 16;

    const uint32_t kMask = opaque_s(0x000F000Fu), kMagic = opaque_v(0x43004300u);
    u32x4 w[2][2];
    u32x2 sreg, breg;
    auto load_w = [&](uint32_t g, u32x4(&r)[2], int q) __attribute__((always_inline)) {
        r[q] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rq, oq + q * 32, g * 64, 2));
    };
    // scale and bias pairs of four steps: lane half h holds steps 2 h, 2 h + 1
    auto load_sb = [&](uint32_t g) {
        sreg = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, os, g * 4, 0));
        breg = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rb, os, g * 4, 0));
    };

    f32x16 acc[MF];
#pragma unroll
    for (int m = 0; m < MF; ++m)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[m][v] = 0.0f;

    // Word j of group gr unpacked to 128 + q (7 VALU)
    auto q_frag = [&](uint32_t q) {
        const u32x4 r = {(q & kMask) | kMagic, ((q >> 4) & kMask) | kMagic, ((q >> 8) & kMask) | kMagic,
                         ((q >> 12) & kMask) | kMagic};
        return __builtin_bit_cast(bf16x8_t, r);
    };
    uint32_t sv, bv;  // the step's scale and bias pairs of the lane's weight row
    auto scales = [&](uint32_t u, uint32_t i) __attribute__((always_inline)) {
        sv = __builtin_amdgcn_ds_bpermute(c * 4 + (i & 2) * 64, sreg[u]);
        bv = __builtin_amdgcn_ds_bpermute(c * 4 + (i & 2) * 64, breg[u]);
    };
    // X and the weights of step i + 1 are requested at step i.  vmcnt completes in issue order, so the wait for X
    // leaves the weight requests in flight.  (Weights three steps ahead: 4-8 % slower; matrix instructions, FMAs and
    // LDS reads pinned in a hand-made order: 10 % slower than the compiler's.)
    auto step = [&](auto U, auto NAc, uint32_t i) __attribute__((always_inline)) {
        constexpr int u = decltype(U)::value, NA = decltype(NAc)::value;
        const uint32_t gn = min(i + 1, GS - 1);
#pragma unroll
        for (int q = 0; q < 2 * NA; ++q) dma_x(gn, u ^ 1, q);  // 2 NA requests cover 32 NA rows
        dma_u(gn, u ^ 1);
        __builtin_amdgcn_sched_barrier(0);
        load_w(gn, w[u ^ 1], 0);
        load_w(gn, w[u ^ 1], 1);
        __builtin_amdgcn_sched_barrier(0);
        const char *xb = lds + u * T::kBuf;
        // the S terms: this lane half's group of b and -128 s against (hi mid lo hi mid lo 0 0) of S
        const uint32_t bh = h ? bv >> 16 : bv & 0xFFFFu;
        const float sh = __uint_as_float(h ? sv & 0xFFFF0000u : sv << 16);
        const uint32_t th = __float_as_uint(sh * -128.0f) >> 16;
        const bf16x8_t bs = __builtin_bit_cast(bf16x8_t, u32x4{bh | (bh << 16), bh | (th << 16), th | (th << 16), 0u});
#pragma unroll
        for (int m = 0; m < NA; ++m)
            acc[m] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8_t *>(xb + ua + m * 1024), bs,
                                                             acc[m], 0, 0, 0);
#pragma unroll
        for (int gr = 0; gr < 2; ++gr) {
            const float sg = __uint_as_float(gr ? sv & 0xFFFF0000u : sv << 16);
            bf16x8_t bf[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) bf[j] = q_frag(w[u][gr][j]);
#pragma unroll
            for (int m = 0; m < NA; ++m) {
                f32x16 d = {};
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        *reinterpret_cast<const bf16x8_t *>(xb + (xa0 ^ ((8 * gr + j) << 4)) + m * 8192), bf[j], d, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[m][v] = fmaf(sg, d[v], acc[m][v]);
            }
        }
        scales(u ^ 1, i + 1);
        asm volatile("s_waitcnt vmcnt(2)" ::: "memory");  // the X step has landed; the newest weights stay in flight
        if constexpr (u == 0) {  // past the last use of the block's scales: the next four steps'
            if (i & 2) load_sb(min(i + 2, GS - 1));
        }
        __syncthreads();
    };
    auto run = [&](auto NAc) __attribute__((always_inline)) {
        uint32_t i = 0;
        for (; i + 2 <= GS; i += 2) {
            step(std::integral_constant<int, 0>{}, NAc, i);
            step(std::integral_constant<int, 1>{}, NAc, i + 1);
        }
        if (i < GS) step(std::integral_constant<int, 0>{}, NAc, i);
    };
#pragma unroll
    for (int q = 0; q < XI; ++q) dma_x(0, 0, q);
    dma_u(0, 0);
    load_sb(0);
    load_w(0, w[0], 0);
    load_w(0, w[0], 1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    scales(0, 0);
    __syncthreads();
    if constexpr (MF == 1) {
        run(std::integral_constant<int, 1>{});
    } else {
        static_assert(MF == 3, "one or three row fragments");
        if (na == 1) run(std::integral_constant<int, 1>{});
        else if (na == 2) run(std::integral_constant<int, 2>{});
        else run(std::integral_constant<int, 3>{});
    }
    // the last step's look-ahead loads have landed before the tile is written over the X buffers
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

    // ---- epilogue, 32 tokens at a time through LDS (a lane holds column c, rows 8 q + 4 h + v of a fragment)
    float *tile = reinterpret_cast<float *>(lds);
    // Non-finite sums (an infinite x, or |x| beyond about 2e36, whose product with 128 + q overflows) are computed
    // again in plain f32: the three parts of an infinite S cannot meet b and -128 s.
    auto finite8 = [](const float *g, int second) {  // 8 sums, and the 8 at + second; 0 times a non-finite one is NaN
        float z = 0.0f;
#pragma unroll
        for (int v = 0; v < 8; ++v) z = fmaf(g[second + v], 0.0f, fmaf(g[v], 0.0f, z));
        return z == z;
    };
    auto exact8 = [&](const Q4Mat &Wm, float *g, uint32_t p, uint32_t n) {
        const uint16_t *xr = reinterpret_cast<const uint16_t *>(a.xp) + (size_t)(a.x_div ? a.sorted[p] / a.x_div : p) * K;
#pragma unroll 1
        for (int v = 0; v < 8; ++v)
            if (!__builtin_isfinite(g[v])) g[v] = q4_exact_dot<true>(Wm, er + n + v, xr, K, 0, K);
    };
    static_for<MF>([&](auto Mi) {
        constexpr int m = Mi;
        if ((uint32_t)m >= na) return;
        __syncthreads();
#pragma unroll
        for (int v = 0; v < 16; ++v)
            tile[(8 * (v >> 2) + 4 * h + (v & 3)) * T::kPitch + wave * 32 + c] = acc[m][v];
        __syncthreads();
        if constexpr (kGateUp) {
            const uint32_t r = (uint32_t)tid >> 3, cu = (uint32_t)tid & 7;
            float *g = tile + r * T::kPitch + cu * 8;
            const uint32_t n = nt * 64 + cu * 8, p = p0 + 32 * m + r;
            const bool live = 32 * m + r < rows && n < a.rows;
            if (live && !finite8(g, 64)) {
                exact8(a.w, g, p, n);
                exact8(a.w2, g + 64, p, n);
            }
            float t[8];
#pragma unroll
            for (int v = 0; v < 8; ++v) t[v] = activation(g[v], a.act) * g[64 + v];
            u32x4 o = {f32_to_bf16(t[0]) | (f32_to_bf16(t[1]) << 16), f32_to_bf16(t[2]) | (f32_to_bf16(t[3]) << 16),
                       f32_to_bf16(t[4]) | (f32_to_bf16(t[5]) << 16), f32_to_bf16(t[6]) | (f32_to_bf16(t[7]) << 16)};
            const float s = group_sum(o);
            if (live) {
                *reinterpret_cast<u32x4 *>(a.out_h + (size_t)p * a.rows + n) = pair_order(o);
                if (cu == 0) a.out_su[(size_t)p * (a.rows >> 6) + nt] = sum_unit(s);
            }
        } else {
#pragma unroll
            for (int it = 0; it < 2; ++it) {
                const uint32_t r = (uint32_t)(tid + 256 * it) >> 4, cu = (uint32_t)tid & 15;
                const uint32_t n = nt * 128 + cu * 8;
                if (32 * m + r < rows && n < a.rows) {
                    float *g = tile + r * T::kPitch + cu * 8;
                    if (!finite8(g, 0)) exact8(a.w, g, p0 + 32 * m + r, n);
                    const f32x4 *src = reinterpret_cast<const f32x4 *>(g);
                    f32x4 *dst = reinterpret_cast<f32x4 *>(a.out_d + (size_t)a.sorted[p0 + 32 * m + r] * a.rows + n);
                    dst[0] = src[0];
                    dst[1] = src[1];
                }
            }
        }
    });
}

template <int MF, bool kGateUp, int OCC>
hipError_t launch_grouped_t(const GroupedArgs &a, hipStream_t s) {
    using T = GroupedTile<MF>;
    constexpr uint32_t kCols = kGateUp ? 64 : 128;
    // an upper bound of the tiles: the buckets are on the device; blocks past the real number exit
    const uint64_t mtiles = (uint64_t)a.assign / T::kBM + std::min(a.experts, a.assign);
    const uint64_t grid = mtiles * ((a.rows + kCols - 1) / kCols);
    if (grid == 0 || grid >= (1ull << 31)) return hipErrorInvalidValue;
    hipLaunchKernelGGL((q4_grouped_kernel<MF, kGateUp, OCC>), dim3((uint32_t)grid), dim3(256), T::kLds, s, a);
    return hipGetLastError();
}

// 32-token tiles (four blocks per CU) or 96-token ones, by moe_wide_tiles() (launch_rules.hpp).  (8 experts, 2000 tokens, top
// 2, the experts' call in us with 32 / 64 / 96 / 128-token tiles: 288 / 223 / 205 / 261; the last spill.)
template <bool kGateUp>
hipError_t launch_grouped_m(const GroupedArgs &a, hipStream_t s) {
    constexpr uint32_t kCols = kGateUp ? 64 : 128;
    if (moe_wide_tiles(a.assign, a.experts, (a.rows + kCols - 1) / kCols, kGateUp, (uint32_t)device_cus()))
        return launch_grouped_t<3, kGateUp, 2>(a, s);
    return launch_grouped_t<1, kGateUp, 4>(a, s);
}

}  // namespace

hipError_t launch_moe_x_prep(const uint16_t *x, uint32_t rows, uint32_t k, void *xp, void *su, hipStream_t s) {
    const uint64_t units = (uint64_t)rows * (k / 8);
    if (k % 128 != 0 || units == 0 || units >= (1ull << 31)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(moe_x_prep_kernel, dim3((uint32_t)((units + 255) / 256)), dim3(256), 0, s,
                       reinterpret_cast<const u32x4 *>(x), reinterpret_cast<u32x4 *>(xp), reinterpret_cast<u32x4 *>(su),
                       (uint32_t)units);
    return hipGetLastError();
}

bool grouped_fits(uint32_t rows, uint32_t k, uint32_t xrows, uint32_t experts, uint32_t assign) {
    return k % 128 == 0 && k != 0 && rows % 64 == 0 && rows != 0 && experts != 0 && experts <= kMaxExperts && assign != 0 &&
           (uint64_t)xrows * k * 2 < (1ull << 32) && (uint64_t)rows * (k / 2) < (1ull << 32) &&
           ((uint64_t)assign / 32 + experts) * (rows / 64) < (1ull << 31);
}

hipError_t launch_grouped(const GroupedArgs &a, hipStream_t s) {
    if (!grouped_fits(a.rows, a.k, a.xrows, a.experts, a.assign)) return hipErrorInvalidValue;
    return a.w2.qw ? launch_grouped_m<true>(a, s) : launch_grouped_m<false>(a, s);
}

}  // namespace kr
