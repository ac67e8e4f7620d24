// q4_prefill.hpp — device helpers shared by the prefill kernels (q4_prefill.hip, q4_prefill_wide.hip):
// buffer resources, direct-to-LDS loads, fp16 operands and the epilogue's stores.
#pragma once

#include "kr_internal.hpp"

namespace kr {

using rsrc_t = __amdgpu_buffer_rsrc_t;

__device__ __forceinline__ rsrc_t make_rsrc(const void *p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)bytes, 0x00020000);
}

__device__ __forceinline__ uint32_t opaque_v(uint32_t v) {
    uint32_t r;
    asm volatile("v_mov_b32 %0, %1" : "=v"(r) : "i"(v));
    return r;
}

__device__ __forceinline__ uint32_t opaque_s(uint32_t v) {
    uint32_t r;
    asm volatile("s_mov_b32 %0, %1" : "=s"(r) : "i"(v));
    return r;
}

__device__ __forceinline__ f16x2_t f16_pair(uint32_t bf16_bits) {
    const _Float16 h = (_Float16)bf16_to_f32(bf16_bits);
    return f16x2_t{h, h};
}

// LDS row swizzle of the X slice: 16 consecutive rows x one unit hit 16
// distinct 16-byte slots modulo 256 bytes, and 8 consecutive rows distinct
// slots modulo 128 bytes.
__device__ __forceinline__ uint32_t swz(uint32_t r) { return (r & 7) ^ ((r >> 3) & 1); }

// 16 bytes per lane from a buffer straight into LDS: lane l writes lds[16 l, 16 l + 16).
// `lds` must be wave-uniform (it goes to M0).
__device__ __forceinline__ void dma16(rsrc_t r, char *lds, uint32_t voffset, uint32_t soffset) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void *)lds, 16, voffset, soffset, 0,
                                             0);
}

// 8 nibbles of one word -> the B fragment (w0 w4)(w1 w5)(w2 w6)(w3 w7), w = fma(q, s, b).
__device__ __forceinline__ f16x8_t dequant_pairs(uint32_t w, f16x2_t s2, f16x2_t b2, uint32_t mask, uint32_t magic) {
    const f16x2_t k1024 = {(_Float16)-1024.0f, (_Float16)-1024.0f};
    f16x2_t pr[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t h = ((w >> (4 * j)) & mask) | magic;           // (1024 + q_j, 1024 + q_{j+4})
        pr[j] = __builtin_elementwise_fma(__builtin_bit_cast(f16x2_t, h) + k1024, s2, b2);
    }
    return f16x8_t{pr[0].x, pr[0].y, pr[1].x, pr[1].y, pr[2].x, pr[2].y, pr[3].x, pr[3].y};
}

// 8 bf16 columns (x0 x1)(x2 x3)(x4 x5)(x6 x7) -> fp16 (x0 x4)(x1 x5)(x2 x6)(x3 x7).
__device__ __forceinline__ u32x4 x_unit_f16(u32x4 d) {
    auto lo = [](uint32_t v) { return __uint_as_float(v << 16); };
    auto hi = [](uint32_t v) { return __uint_as_float(v & 0xFFFF0000u); };
    const f16x2_t o0 = {(_Float16)lo(d.x), (_Float16)lo(d.z)};
    const f16x2_t o1 = {(_Float16)hi(d.x), (_Float16)hi(d.z)};
    const f16x2_t o2 = {(_Float16)lo(d.y), (_Float16)lo(d.w)};
    const f16x2_t o3 = {(_Float16)hi(d.y), (_Float16)hi(d.w)};
    return u32x4{__builtin_bit_cast(uint32_t, o0), __builtin_bit_cast(uint32_t, o1),
                 __builtin_bit_cast(uint32_t, o2), __builtin_bit_cast(uint32_t, o3)};
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

}  // namespace kr
