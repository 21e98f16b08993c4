// Device helpers of the fused passes (fused.hip) and of the lifts in keyswitch.hip.
#pragma once
#include "fused.hpp"
#include "row_tile.hpp"

namespace ck {

// Loads at a uniform pointer plus a 32-bit byte offset per lane: one register
// of address per lane instead of a 64-bit pointer per load.
__device__ __forceinline__ u64 load_at(const u64 *base, u32 byte_off) {
    return *(const u64 *)((const char *)base + byte_off);
}
__device__ __forceinline__ u64 load_once_at(const u64 *base, u32 byte_off) {
    return ld_stream((const u64 *)((const char *)base + byte_off));
}
__device__ __forceinline__ void store_once_at(u64 *base, u32 byte_off, u64 v) {
    st_stream((u64 *)((char *)base + byte_off), v);
}
__device__ __forceinline__ double load_z(const double *base, u32 off) {
    return *(const double *)((const char *)base + off * 8);
}
__device__ __forceinline__ Tw load_z(const Tw *base, u32 off) { return *(const Tw *)((const char *)base + off * 16); }
// two residues; callers' strides leave 8-byte alignment only
typedef u64 u64x2 __attribute__((ext_vector_type(2), aligned(8)));
__device__ __forceinline__ u64x2 load2_at(const u64 *base, u32 byte_off) {
    return *(const u64x2 *)((const char *)base + byte_off);
}

// A value the compiler cannot see through: index math that depends on it
// stays inside the digit loop instead of being kept in registers across it.
__device__ __forceinline__ u32 opaque(u32 x) {
#if defined(__HIP_DEVICE_COMPILE__)
    asm volatile("" : "+v"(x));
#endif
    return x;
}

// 2^52 + 2^51 + d in the mantissa: exact for |d| < 2^51
__device__ __forceinline__ double signed_to_f64(u64 d) {
    return u64_as_f64(d + 0x4338000000000000ull) - 6755399441055744.0;
}

// The value sum_t c_t W_t mod q of a gadget block for this thread's residues,
// its digits c_t < 2^41 read from L2 once per target limb instead of the lifted
// value from HBM.  The quotient k = rint(sum_t c_t (W_t / q)) is right to within
// one (c_t exact, W_t / q to 2^-53, at most 13 terms below 2^41, partial sums
// below 2^45: |error| < 0.04), so r = sum_t c_t W_t - k q has |r| < 0.54 q and
// only its low bits are formed: 56 of them for FP64 limbs (one 32x32 product
// and two full-rate 24-bit cross products a term), 64 for integer limbs.  With
// the FP64 FMA of the quotient an FP64 limb's term takes 14 issue cycles (and
// 7 to convert c_t) where an exact FP64 product takes 31.
// a * b + c of the low 24 bits of a and b (full rate; b uniform).  Written out
// because the compiler, seeing that only low bits of the sum matter, drops the
// 24-bit masks and issues the slow 32-bit product.
__device__ __forceinline__ u32 mad24(u32 a, u32 b, u32 c) {
#if defined(__HIP_DEVICE_COMPILE__)
    u32 r;
    asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
    return r;
#else
    return (a & 0xffffffu) * (b & 0xffffffu) + c;
#endif
}

// A digit c < 2^41 as the bits of the double 2^52 + c: its low word is c's, its
// high word c's with the exponent above bit 20.
constexpr u64 kDigitBias = 0x4330000000000000ull;

template <bool FP>
struct BlockSum {
    double k = 0.0;
    u32 lo = 0, hi = 0;
    // a b + c of high-word parts: FP64 limbs keep 20 bits of the high word, on
    // which the exponent bits of a biased digit have no effect
    __device__ __forceinline__ static u32 cross(u32 a, u32 b, u32 c) { return FP ? mad24(a, b, c) : a * b + c; }
    __device__ __forceinline__ void add(u64 biased, u64 w, double wp) {
        const u32 c0 = (u32)biased, w0 = (u32)w, w1 = (u32)(w >> 32);
        u32 c1 = (u32)(biased >> 32);
        if (!FP) c1 &= 0xfffffu;
        k = __builtin_fma(u64_as_f64(biased) - 4503599627370496.0, wp, k);
        const u64 p = (u64)c0 * w0 + (((u64)hi << 32) | lo);
        lo = (u32)p;
        hi = cross(c0, w1, cross(c1, w0, (u32)(p >> 32)));
    }
    __device__ __forceinline__ u64 value(u64 q) const {
        const u64 kk = f64_as_u64(__builtin_rint(k) + 4503599627370496.0);  // k in the low 52 bits
        const u32 k0 = (u32)kk, k1 = (u32)(kk >> 32) & 0xfffffu, q0 = (u32)q, q1 = (u32)(q >> 32);
        const u64 d = (((u64)hi << 32) | lo) - (u64)k0 * q0;
        const u32 top = (u32)(d >> 32) - cross(k0, q1, cross(k1, q0, 0));
        if (!FP) return (((u64)top << 32) | (u32)d) + q;  // in (0.4 q, 1.6 q)
        // r mod 2^52 with its sign bit flipped, in the mantissa of 2^52 + ..
        const u32 m = ((top & 0xfffffu) ^ 0x80000u) | 0x43300000u;
        return f64_as_u64(u64_as_f64(((u64)m << 32) | (u32)d) - 6755399441055744.0);
    }
};

// Integer limbs cost two to three times an FP64 limb: they are spread evenly
// among the others, one first, so that heavy and light blocks run side by
// side.  Plans of more limbs run them in order.
constexpr u32 kMaxOrder = 64;

static void limb_order(const ckks_rns_plan *plan, size_t limbs, unsigned char *order) {
    if (limbs > kMaxOrder) return;
    std::vector<unsigned char> heavy, light;
    for (size_t i = 0; i < limbs; ++i) (plan->h_primes[i].fp ? light : heavy).push_back((unsigned char)i);
    size_t h = 0, l = 0;
    for (size_t n = 0; n < limbs; ++n) {
        const bool take = h < heavy.size() && (l >= light.size() || h * light.size() <= l * heavy.size());
        order[n] = take ? heavy[h++] : light[l++];
    }
}

}  // namespace ck
