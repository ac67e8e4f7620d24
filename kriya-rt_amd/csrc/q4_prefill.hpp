// q4_prefill.hpp — device helpers shared by the prefill kernels (q4_prefill.hip, q4_prefill_wide.hip), the grouped
// products (q4_grouped.hip) and the norm that writes their operand (e2e_glue.hip): buffer resources, direct-to-LDS
// loads and fp16 operands.
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

}  // namespace kr
