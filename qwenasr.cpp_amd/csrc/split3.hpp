// The exact three-part bf16 split of an f32 value, for device code only.
//
// v = hi + mid + lo exactly: hi is v cut to 8 significant bits, mid the remainder cut likewise, lo the last remainder,
// which has at most 8 significant bits and so is its own high half.  The row layout (store_split3) truncates, the
// fragment order (split3_pair) rounds to nearest.  Every product of a bf16 weight with one part is exact in f32, which
// is how the prefill GEMMs on bf16-exact weights reproduce f32 products on bf16 MFMA.
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

// The three parts of a and b as pairs of bf16 bits (a low, b high), hi and mid rounded to nearest: |mid| <= 2^-8 |v|,
// |lo| <= 2^-17 |v|, of either sign, so that the products of parts that a GEMM on two split operands leaves out (mid lo,
// lo mid, lo lo) stay within 2^-24 of the whole and do not add up (truncated parts share v's sign and left out up to 2^-21
// of it, always towards zero).  A finite value past the largest bf16 takes that as hi: its parts are exact too.  An
// infinity is 0, 0, itself: the last part meets only the leading part of the other operand, which is zero for a zero
// alone, so its products are those of an f32 GEMM (as the leading part it would meet parts that are zero: NaN).
__device__ inline void split3_pair(float a, float b, uint32_t & hi, uint32_t & mid, uint32_t & lo) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    auto pack = [](float x, float y) {
        const bf16x2 p = {static_cast<__bf16>(x), static_cast<__bf16>(y)};
        return __builtin_bit_cast(uint32_t, p);
    };
    auto low = [](uint32_t p) { return __uint_as_float(p << 16); };
    auto high = [](uint32_t p) { return __uint_as_float(p & 0xffff0000u); };
    constexpr float kMax = 0x1.fep127f;
    const bool ia = __builtin_isinf(a), ib = __builtin_isinf(b);
    hi = pack(ia ? 0.0f : __builtin_amdgcn_fmed3f(a, -kMax, kMax), ib ? 0.0f : __builtin_amdgcn_fmed3f(b, -kMax, kMax));
    a -= low(hi);
    b -= high(hi);
    mid = pack(ia ? 0.0f : a, ib ? 0.0f : b);
    lo = pack(a - low(mid), b - high(mid));
}

// Inputs of the prompt GEMM are stored negated where this holds, in blocks + - - + of kSplitSign k (gemm_prefill.hip says
// what for).
constexpr int kSplitSign = 256;
__device__ inline bool split_negated(int k) { return ((k / kSplitSign ^ k / (2 * kSplitSign)) & 1) != 0; }

// 8 consecutive k (octet o) of row r into the fragment order of an MFMA operand: 32 rows x 16 k of one part are
// 512 consecutive values, lane l = row % 32 + 32 (k / 8 % 2) holding k % 8 = 0..7; fragments follow each other by
// part (hi, mid, lo), then k / 16, then row / 32.  INPUT: negated where split_negated.
template <bool INPUT>
__device__ inline void store_frag8(uint16_t * out, int k16, int r, int o, const float (&v)[8]) {
    const uint32_t sign = INPUT && split_negated(8 * o) ? 0x80008000u : 0u;
    uint32_t part[3][4];
#pragma unroll
    for (int e = 0; e < 4; ++e) split3_pair(v[2 * e], v[2 * e + 1], part[0][e], part[1][e], part[2][e]);
    uint16_t * d = out + (static_cast<int64_t>(r >> 5) * k16 + (o >> 1)) * 3 * 512 + ((r & 31) + 32 * (o & 1)) * 8;
#pragma unroll
    for (int w = 0; w < 3; ++w) {
        *reinterpret_cast<uint4 *>(d + w * 512) = make_uint4(part[w][0] ^ sign, part[w][1] ^ sign, part[w][2] ^ sign, part[w][3] ^ sign);
    }
}

// 4 consecutive k (first k % 4 == 0) of row r of an input into the same order
__device__ inline void store_frag4(uint16_t * out, int k16, int r, int k, float v0, float v1, float v2, float v3) {
    const uint32_t sign = split_negated(k) ? 0x80008000u : 0u;
    uint32_t part[3][2];
    split3_pair(v0, v1, part[0][0], part[1][0], part[2][0]);
    split3_pair(v2, v3, part[0][1], part[1][1], part[2][1]);
    uint16_t * d = out + (static_cast<int64_t>(r >> 5) * k16 + (k >> 4)) * 3 * 512 + ((r & 31) + 32 * ((k >> 3) & 1)) * 8 + (k & 7);
#pragma unroll
    for (int w = 0; w < 3; ++w) *reinterpret_cast<uint2 *>(d + w * 512) = make_uint2(part[w][0] ^ sign, part[w][1] ^ sign);
}

}  // namespace qa
