// LDS rows read as 128-bit vectors, shared by the plane-marching kernels.
#pragma once
#include "lncc_common.h"

namespace fl {

// A row of NV consecutive floats at a 16-byte aligned LDS address, read as float4s, then a tail of 2
// or 1 floats as a float2 or a float (a tail of 3 as one more float4, which reads one float past the
// row; it is not used), row_read(NV) floats in all. row_load issues the reads; row_take hands out the
// values, each vector through an empty asm operand that needs all of its lanes, so that the loads
// stay whole: otherwise the optimizer re-partitions them along the box-sums' blocks (a row of 10
// floats became b128 + b96 + read2_b32 + b32 instead of b128 + b128 + b64), which costs LDS
// instructions and bank cycles. The operand is a use, so the wait for the reads stands where row_take
// stands: behind the work that is to cover their latency, not behind the reads. The 2-float tail
// (rather than a third float4) also keeps two registers per row free.
typedef float lds_f4 __attribute__((ext_vector_type(4)));
typedef float lds_f2 __attribute__((ext_vector_type(2)));
// the vectors of such a row: NQ float4s, then one float2 if there is a tail of 1 or 2
FL_HD constexpr int row_quads(int n) { return row_read(n) / 4; }
template <int NV>
__device__ __forceinline__ void row_load(const float* __restrict__ src, lds_f4* q, lds_f2& h) {
    static_assert(row_read(NV) >= NV && row_quads(NV) * 4 <= row_read(NV), "row read");
#pragma unroll
    for (int m = 0; m < row_quads(NV); ++m) q[m] = reinterpret_cast<const lds_f4*>(src)[m];
    constexpr int t = row_quads(NV) * 4;
    if constexpr (NV - t == 2) h = *reinterpret_cast<const lds_f2*>(src + t);
    if constexpr (NV - t == 1) h.x = src[t];
}
template <int NV>
__device__ __forceinline__ void row_take(const lds_f4* q, const lds_f2& h, float (&v)[NV]) {
#pragma unroll
    for (int m = 0; m < row_quads(NV); ++m) {
        lds_f4 f = q[m];
        asm("" : "+v"(f));
        v[4 * m] = f.x;
        v[4 * m + 1] = f.y;
        v[4 * m + 2] = f.z;
        if (4 * m + 3 < NV) v[4 * m + 3 < NV ? 4 * m + 3 : 0] = f.w;
    }
    constexpr int t = row_quads(NV) * 4;
    if constexpr (NV - t == 2) {
        lds_f2 f = h;
        asm("" : "+v"(f));
        v[t] = f.x;
        v[t + 1] = f.y;
    }
    if constexpr (NV - t == 1) {
        float f = h.x;
        asm("" : "+v"(f));
        v[t] = f;
    }
}
template <int NV>
__device__ __forceinline__ void lds_row(const float* __restrict__ src, float (&v)[NV]) {
    lds_f4 q[row_quads(NV)];
    lds_f2 h;
    row_load<NV>(src, q, h);
    row_take<NV>(q, h, v);
}

// Stores four floats to a 16-byte aligned LDS address as one 128-bit write. The vector passes
// through an empty asm operand that needs all of its lanes, for the reason given at lds_row: left
// alone, the compiler split the AYs stores into pairs of adjacent 32-bit writes (ds_write2_b32),
// and at the row stride of GY (36 floats) each such write served 64 lanes from 16 banks, 4-way
// conflicts: a quarter of the kernel's LDS bank-conflict cycles came from them.
__device__ __forceinline__ void lds_store4(float* __restrict__ dst, float x, float y, float z, float w) {
    lds_f4 f = {x, y, z, w};
    asm("" : "+v"(f));
    *reinterpret_cast<lds_f4*>(dst) = f;
}

}  // namespace fl
