// The exact three-part bf16 split of an f32 value, for device code only.
//
// v = hi + mid + lo exactly: hi is v truncated to its top 8 significant bits (the high half of its bits),
// mid the same truncation of the remainder, lo the last remainder, which has at most 8 significant bits
// and so is its own high half.  Every product of a bf16 weight with one part is exact in f32, which is how
// the prefill GEMMs on bf16-exact weights reproduce f32 products on bf16 MFMA.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace qa {

// the three parts of v as bf16 bits at o[0], o[K], o[2 K]: the layout of one row of a split GEMM input
__device__ inline void store_split3(uint16_t * o, int64_t K, float v) {
    const uint32_t h = __float_as_uint(v) & 0xffff0000u;
    const float r1 = v - __uint_as_float(h);
    const uint32_t m = __float_as_uint(r1) & 0xffff0000u;
    const float r2 = r1 - __uint_as_float(m);
    o[0] = static_cast<uint16_t>(h >> 16);
    o[K] = static_cast<uint16_t>(m >> 16);
    o[2 * K] = static_cast<uint16_t>(__float_as_uint(r2) >> 16);
}

// the three parts of v as bf16 bits.  An infinity is 0, 0, itself: the last part meets only the leading part of the
// other operand, which is zero for a zero alone, so its products are those of an f32 GEMM (as the leading part it would
// meet parts that are zero, and infinity times zero is NaN).
__device__ inline void split3_parts(float v, uint16_t & hi, uint16_t & mid, uint16_t & lo) {
    const bool inf = __builtin_isinf(v);
    const uint32_t h = inf ? 0u : __float_as_uint(v) & 0xffff0000u;
    const float r1 = v - __uint_as_float(h);
    const uint32_t m = inf ? 0u : __float_as_uint(r1) & 0xffff0000u;
    hi = static_cast<uint16_t>(h >> 16);
    mid = static_cast<uint16_t>(m >> 16);
    lo = static_cast<uint16_t>(__float_as_uint(r1 - __uint_as_float(m)) >> 16);
}

// 8 consecutive k (octet o) of row r into the fragment order of an MFMA operand: 32 rows x 16 k of one part are
// 512 consecutive values, lane l = row % 32 + 32 (k / 8 % 2) holding k % 8 = 0..7; fragments follow each other by
// part (hi, mid, lo), then k / 16, then row / 32.
__device__ inline void store_frag8(uint16_t * out, int k16, int r, int o, const float (&v)[8]) {
    uint16_t part[3][8];
#pragma unroll
    for (int e = 0; e < 8; ++e) split3_parts(v[e], part[0][e], part[1][e], part[2][e]);
    uint16_t * d = out + (static_cast<int64_t>(r >> 5) * k16 + (o >> 1)) * 3 * 512 + ((r & 31) + 32 * (o & 1)) * 8;
#pragma unroll
    for (int w = 0; w < 3; ++w) {
        uint4 u;
        u.x = part[w][0] | (static_cast<uint32_t>(part[w][1]) << 16);
        u.y = part[w][2] | (static_cast<uint32_t>(part[w][3]) << 16);
        u.z = part[w][4] | (static_cast<uint32_t>(part[w][5]) << 16);
        u.w = part[w][6] | (static_cast<uint32_t>(part[w][7]) << 16);
        *reinterpret_cast<uint4 *>(d + w * 512) = u;
    }
}

// 4 consecutive k (first k % 4 == 0) of row r into the same order
__device__ inline void store_frag4(uint16_t * out, int k16, int r, int k, float v0, float v1, float v2, float v3) {
    const float v[4] = {v0, v1, v2, v3};
    uint16_t part[3][4];
#pragma unroll
    for (int e = 0; e < 4; ++e) split3_parts(v[e], part[0][e], part[1][e], part[2][e]);
    uint16_t * d = out + (static_cast<int64_t>(r >> 5) * k16 + (k >> 4)) * 3 * 512 + ((r & 31) + 32 * ((k >> 3) & 1)) * 8 + (k & 7);
#pragma unroll
    for (int w = 0; w < 3; ++w) {
        *reinterpret_cast<uint2 *>(d + w * 512) = make_uint2(part[w][0] | (static_cast<uint32_t>(part[w][1]) << 16),
                                                             part[w][2] | (static_cast<uint32_t>(part[w][3]) << 16));
    }
}

}  // namespace qa
