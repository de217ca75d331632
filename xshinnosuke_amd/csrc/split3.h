// A float32 as the exact sum of three bf16 values (conv_split.hip says what that is good for).
#pragma once
#include "xsmi_internal.h"

#include <type_traits>

namespace xsmi {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t uint32x4 __attribute__((ext_vector_type(4)));

template <int N>
using IC = std::integral_constant<int, N>;

// two floats -> bf16 pair (nearest even); the pair's values taken off the floats (v_dot2_f32_bf16 with (-1, 0) and (0, -1): one
// instruction for a subtraction and the widening in front of it; the difference is representable, so it is exact)
__device__ __forceinline__ uint32_t split_pair(float &a, float &b) {
    const bf16x2 p = {(__bf16)a, (__bf16)b}, hi = {(__bf16)0.f, (__bf16)-1.f};
    uint32_t lo_bits = 0x0000bf80u;                            // (-1, 0), kept from the compiler: as an inline constant -1.0
    asm("" : "+s"(lo_bits));                                   // it comes out as (0, -1)
    const bf16x2 lo = __builtin_bit_cast(bf16x2, lo_bits);
    a = __builtin_amdgcn_fdot2_f32_bf16(p, lo, a, false);
    b = __builtin_amdgcn_fdot2_f32_bf16(p, hi, b, false);
    return __builtin_bit_cast(uint32_t, p);
}

// two floats -> the three bf16 pairs of their split
__device__ __forceinline__ void split_pair3(float a, float b, uint32_t &p0, uint32_t &p1, uint32_t &p2) {
    p0 = split_pair(a, b);
    p1 = split_pair(a, b);
    const bf16x2 l = {(__bf16)a, (__bf16)b};
    p2 = __builtin_bit_cast(uint32_t, l);
}

// Which values have a split.  Infinities, NaN and values that round to a bf16 infinity make every sum they enter a NaN by
// themselves.  Values below 2^-110 lose bits instead: the last piece ends at 2^-133, the smallest bf16 (3 x 3, 64 channels,
// values of 2^-112: 1.6e-7 against 64 bits, of 2^-124: 5.7e-4, of 2^-136: everything; fp32 pipe 1.1e-7), whatever the other
// operand is.  The kernels look for them while they split and put a NaN in the first piece.
constexpr uint32_t NAN_PAIR = 0x7fc07fc0u;
struct SmallTest {                                     // one and a half instructions a value
    uint32_t smallest = 0xffffffffu;                   // twice a value's bits without the sign, less one: zero is the largest
    __device__ __forceinline__ void add(float a, float b) {
        const uint32_t x = __builtin_bit_cast(uint32_t, a) * 2u - 1u, y = __builtin_bit_cast(uint32_t, b) * 2u - 1u;
        smallest = x < smallest ? x : smallest;
        smallest = y < smallest ? y : smallest;
    }
    __device__ __forceinline__ bool found() const { return smallest < 2u * 0x08800000u - 1u; }
};
static_assert(__builtin_bit_cast(float, 0x08800000u) == 0x1p-110f, "the bits of 2^-110");
__device__ __forceinline__ bool splits(float v) {
    const float a = __builtin_fabsf(v);
    return a < __builtin_bit_cast(float, 0x7f7f8000u) && (a >= 0x1p-110f || a == 0.f);
}
struct SplitTest {                                     // whether many values all split, three instructions a value
    uint32_t smallest = 0xffffffffu, largest = 0;      // of twice the bits without the sign, the smallest less one
    __device__ __forceinline__ void add(float v) {
        const uint32_t x = __builtin_bit_cast(uint32_t, v) * 2u, m = x - 1u;
        smallest = m < smallest ? m : smallest;
        largest = x > largest ? x : largest;
    }
    __device__ __forceinline__ bool all() const { return smallest >= 2u * 0x08800000u - 1u && largest < 2u * 0x7f7f8000u; }
};

// Whether a sum of split products is as good as the float32 one.  It is not if an operand had no split (the sum is then a NaN
// or infinite).  Sums below 2^-100 are formed again as well: their small products run out of bits, as the fp32 pipe's do
// (2^-66 times 2^-66: 2.7e-5 against 64 bits, fp32 pipe 4.4e-5, formed again 3.8e-6).
__device__ __forceinline__ bool carried(float v) {
    const float a = __builtin_fabsf(v);
    return a < __builtin_inff() && (a >= 0x1p-100f || a == 0.f);
}
// The same for many values, at two and a half instructions each.
struct CarriedTest {
    float zero = 0.f;                                  // NaN from an infinity or a NaN on
    uint32_t smallest = 0xffffffffu;                   // twice a value's bits without the sign, less one: zero is the largest
    __device__ __forceinline__ void add(float v) {
        zero = __builtin_fmaf(v, 0.f, zero);
        const uint32_t m = __builtin_bit_cast(uint32_t, v) * 2u - 1u;
        smallest = m < smallest ? m : smallest;
    }
    __device__ __forceinline__ bool all() const { return zero == 0.f && smallest >= 2u * 0x0d800000u - 1u; }
};
static_assert(__builtin_bit_cast(float, 0x0d800000u) == 0x1p-100f, "the bits of 2^-100");

// The sums of a 32 x 32 block (register v of lane l is row 8 (v / 4) + 4 (l / 32) + v % 4, column l % 32) that are not carried, formed
// in float64: four 16 x 16 blocks on the fp64 matrix instruction (D: register k of lane l is row l / 16 + 4 k, column l % 16).
// Blocks that have no such sum are left out, and a sum that has become a NaN stays one: once all of them have, the terms that
// are left are not read.  A tensor that holds NaN throughout then costs its first terms instead of all.
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef double doublex4 __attribute__((ext_vector_type(4)));
struct FormAgain {
    doublex4 d[2][2];                                  // [rows][columns]
    uint32_t need;                                     // bit 8 i + 4 (k / 2) + 2 (k % 2) + j for register k of rows i, columns j
    uint32_t use;                                      // bit 2 i + j: whether any lane needs the block
    // every sum of the columns that are there, in short code: what a kernel rarely does it also fetches for the occasion
    __device__ __forceinline__ FormAgain(bool column_there, int lane) : need(0), use(15) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            need |= __shfl((int)column_there, 16 * j + (lane & 15)) ? 0x5555u << j : 0u;
            d[0][j] = d[1][j] = doublex4{0.0, 0.0, 0.0, 0.0};
        }
    }
    // those that are not carried, for long sums
    __device__ __forceinline__ FormAgain(const floatx16 &r, bool column_there, int lane) : need(0), use(0) {
        uint32_t open = 0;
#pragma unroll
        for (int v = 0; v < 16; ++v) open |= (carried(r[v]) ? 0u : 1u) << v;
        open = column_there ? open : 0u;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            need |= (((uint32_t)__shfl((int)open, 32 * (i >> 1) + 16 * (i & 1) + (lane & 15)) >> (lane >> 4)) & 0x1111u) << i;
            d[i >> 1][i & 1] = doublex4{0.0, 0.0, 0.0, 0.0};
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) use |= (__builtin_amdgcn_ballot_w64((need & (0x55u << (8 * (i >> 1) + (i & 1)))) != 0) != 0 ? 1u : 0u) << i;
    }
    __device__ __forceinline__ void add(const double (&a)[2], const double (&b)[2]) {   // four terms
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (use >> i & 1) d[i >> 1][i & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i >> 1], b[i & 1], d[i >> 1][i & 1], 0, 0, 0);
    }
    __device__ __forceinline__ bool settled() const {
        uint32_t open = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const double v = d[i >> 1][i & 1][k];
                open |= v == v ? need & (1u << (8 * (i >> 1) + 4 * (k >> 1) + 2 * (k & 1) + (i & 1))) : 0u;
            }
        return __builtin_amdgcn_ballot_w64(open != 0) == 0;
    }
    __device__ __forceinline__ void take(floatx16 &r, int lane) const {
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            float from[2][2];                          // [right half of the columns][upper half of the lanes]
#pragma unroll
            for (int k = 0; k < 4; ++k)
                from[k >> 1][k & 1] = __shfl((float)d[v >> 3][k >> 1][2 * ((v >> 2) & 1) + (k & 1)], 16 * (v & 3) + (lane & 15));
            const float low = (lane & 16) ? from[1][0] : from[0][0], high = (lane & 16) ? from[1][1] : from[0][1];
            const float again = (lane & 32) ? high : low;
            r[v] = carried(r[v]) ? r[v] : again;
        }
    }
};

}  // namespace xsmi
