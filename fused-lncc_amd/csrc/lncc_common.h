// Shared device helpers for the gfx950 LNCC kernels: buffer resources, bf16 conversion, tile
// geometry. Included by the kernel translation units only.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "lncc_geometry.h"

namespace fl {

// gfx9 buffer resource word 3 (raw buffer, 32-bit data format); out-of-range loads return 0 and
// out-of-range stores are dropped, which gives the zero padding of the box window for free.
constexpr int kRsrcWord3 = 0x00020000;
constexpr uint32_t kOOB = 0x80000000u;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const void* base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, kRsrcWord3);
}

// The same resource as four plain words, for addresses that advance in place: word 0-1 the address
// (its upper 16 bits are zero for a device address, which is the stride field of a raw buffer),
// word 2 the size in bytes (0: loads return 0, stores are dropped), word 3 as above. Built this way
// a plane's resource costs the two scalar additions that advance its address; through
// make_buffer_rsrc the compiler masks the address and rebuilds all four words for every access.
typedef int rsrc_words __attribute__((ext_vector_type(4)));
__device__ __forceinline__ rsrc_words words_at(uint64_t addr, uint32_t bytes) {
    return rsrc_words{(int)(uint32_t)addr, (int)(uint32_t)(addr >> 32), (int)bytes, kRsrcWord3};
}
__device__ float raw_load_f32(rsrc_words r, int voff, int soff, int aux) __asm("llvm.amdgcn.raw.buffer.load.f32");
typedef float f32x3 __attribute__((ext_vector_type(3)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
__device__ f32x3 raw_load_f32x3(rsrc_words r, int voff, int soff, int aux) __asm("llvm.amdgcn.raw.buffer.load.v3f32");
__device__ f32x4 raw_load_f32x4(rsrc_words r, int voff, int soff, int aux) __asm("llvm.amdgcn.raw.buffer.load.v4f32");
__device__ unsigned short raw_load_b16(rsrc_words r, int voff, int soff, int aux) __asm("llvm.amdgcn.raw.buffer.load.i16");
__device__ void raw_store_f32(float v, rsrc_words r, int voff, int soff, int aux) __asm("llvm.amdgcn.raw.buffer.store.f32");
__device__ void raw_store_b16(unsigned short v, rsrc_words r, int voff, int soff, int aux) __asm("llvm.amdgcn.raw.buffer.store.i16");

// Cache-policy operand of the buffer instructions: 0 = default, kNT = non-temporal (the line is
// streamed: a store does not displace data that will be read again from the L2, a load marks the
// line as the first to evict).
constexpr int kNT = 2;

template <bool BF16, int AUX = 0>
__device__ __forceinline__ float load_elem(__amdgpu_buffer_rsrc_t r, uint32_t voff) {
    if constexpr (BF16) {
        uint32_t u = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(r, (int)voff, 0, AUX);
        return __uint_as_float(u << 16);
    } else {
        // the builtin returns the raw 32 bits; reinterpret, do not convert
        return __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, (int)voff, 0, AUX));
    }
}

template <bool BF16, int AUX = 0>
__device__ __forceinline__ float load_elem(rsrc_words r, uint32_t voff) {
    if constexpr (BF16)
        return __uint_as_float((uint32_t)raw_load_b16(r, (int)voff, 0, AUX) << 16);
    else
        return raw_load_f32(r, (int)voff, 0, AUX);
}

// The same load for a value that is used a step later: what the load leaves in its register (with
// LATE, a bfloat16's bits), and the float it stands for. load_elem's conversion of a bfloat16 stands
// where the load stands as far as the compiler is concerned, which then waits for the load at the end
// of the step that issued it.
template <bool LATE>
using elem_raw = std::conditional_t<LATE, unsigned short, float>;
template <bool BF16, bool LATE, int AUX = 0>
__device__ __forceinline__ elem_raw<LATE> load_raw(rsrc_words r, uint32_t voff) {
    static_assert(BF16 || !LATE, "float32 needs no conversion");
    if constexpr (LATE)
        return raw_load_b16(r, (int)voff, 0, AUX);
    else
        return load_elem<BF16, AUX>(r, voff);
}
__device__ __forceinline__ float widen(unsigned short bits) {
    asm("" : "+v"(bits));   // here, not at the load
    return __uint_as_float((uint32_t)bits << 16);
}
__device__ __forceinline__ float widen(float v) { return v; }

// N = 3 or 4 consecutive floats in one load (4-byte aligned)
template <int N>
__device__ __forceinline__ void load_run(rsrc_words r, uint32_t voff, float (&v)[N]) {
    static_assert(N == 3 || N == 4, "runs");
    if constexpr (N == 3) {
        const f32x3 f = raw_load_f32x3(r, (int)voff, 0, 0);
        v[0] = f.x, v[1] = f.y, v[2] = f.z;
    } else {
        const f32x4 f = raw_load_f32x4(r, (int)voff, 0, 0);
        v[0] = f.x, v[1] = f.y, v[2] = f.z, v[3] = f.w;
    }
}

template <bool BF16>
__device__ __forceinline__ float load_elem_ptr(const void* base, int64_t idx) {
    if constexpr (BF16) {
        return __uint_as_float((uint32_t)reinterpret_cast<const uint16_t*>(base)[idx] << 16);
    } else {
        return reinterpret_cast<const float*>(base)[idx];
    }
}

// float32 -> bfloat16 bits, round to nearest even; NaN stays a NaN. gfx950 converts in one
// instruction (v_cvt_pk_bf16_f32), which the compiler selects for the __bf16 conversion.
__device__ __forceinline__ uint16_t f32_to_bf16_bits(float x) {
    return __builtin_bit_cast(uint16_t, (__bf16)x);
}

template <bool BF16, int AUX = 0>
__device__ __forceinline__ void store_elem_buf(__amdgpu_buffer_rsrc_t r, uint32_t voff, float v) {
    if constexpr (BF16) {
        __builtin_amdgcn_raw_buffer_store_b16((unsigned short)f32_to_bf16_bits(v), r, (int)voff, 0, AUX);
    } else {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, (int)voff, 0, AUX);
    }
}

template <bool BF16, int AUX = 0>
__device__ __forceinline__ void store_elem_buf(rsrc_words r, uint32_t voff, float v) {
    if constexpr (BF16)
        raw_store_b16(f32_to_bf16_bits(v), r, (int)voff, 0, AUX);
    else
        raw_store_f32(v, r, (int)voff, 0, AUX);
}

template <bool BF16>
__device__ __forceinline__ void store_elem(void* base, int64_t idx, float v) {
    if constexpr (BF16) {
        reinterpret_cast<uint16_t*>(base)[idx] = f32_to_bf16_bits(v);
    } else {
        reinterpret_cast<float*>(base)[idx] = v;
    }
}

// Compile-time loop: f(std::integral_constant<int, I>) for I in [B, E), so that register arrays
// indexed by I stay in registers.
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}

}  // namespace fl
