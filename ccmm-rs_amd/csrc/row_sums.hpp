// Sums of products of the fused passes: gadget blocks from their mixed-radix
// digits, and key products.
#pragma once
#include "row_tile.hpp"

namespace ck {

// 2^52 + 2^51 + d in the mantissa: exact for |d| < 2^51
CK_HD double signed_to_f64(u64 d) {
    return u64_as_f64(d + 0x4338000000000000ull) - 6755399441055744.0;
}

// a * b + c of the low 24 bits of a and b (full rate; b uniform).  Written out
// because the compiler, seeing that only low bits of the sum matter, drops the
// 24-bit masks and issues the slow 32-bit product.
CK_HD u32 mad24(u32 a, u32 b, u32 c) {
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

// The value sum_t c_t W_t mod q of a gadget block for this thread's residues,
// its digits c_t < 2^41 read from L2 once per target limb instead of the lifted
// value from HBM.  The quotient k = rint(sum_t c_t (W_t / q)) is right to within
// one (c_t exact, W_t / q to 2^-53, at most 13 terms below 2^41, partial sums
// below 2^45: |error| < 0.04), so r = sum_t c_t W_t - k q has |r| < 0.54 q and
// only its low bits are formed: 56 of them for FP64 limbs (one 32x32 product
// and two full-rate 24-bit cross products a term), 64 for integer limbs.  With
// the FP64 FMA of the quotient an FP64 limb's term takes 14 issue cycles (and
// 7 to convert c_t) where an exact FP64 product takes 31.
template <bool FP>
struct BlockSum {
    double k = 0.0;
    u32 lo = 0, hi = 0;
    // a b + c of high-word parts: FP64 limbs keep 20 bits of the high word, on
    // which the exponent bits of a biased digit have no effect
    CK_HD static u32 cross(u32 a, u32 b, u32 c) { return FP ? mad24(a, b, c) : a * b + c; }
    CK_HD void add(u64 biased, u64 w, double wp) {
        const u32 c0 = (u32)biased, w0 = (u32)w, w1 = (u32)(w >> 32);
        u32 c1 = (u32)(biased >> 32);
        if (!FP) c1 &= 0xfffffu;
        k = __builtin_fma(u64_as_f64(biased) - 4503599627370496.0, wp, k);
        const u64 p = (u64)c0 * w0 + (((u64)hi << 32) | lo);
        lo = (u32)p;
        hi = cross(c0, w1, cross(c1, w0, (u32)(p >> 32)));
    }
    CK_HD u64 value(u64 q) const {
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

// Two sums per residue, 64 bits each.
//   FP64: products within 0.52 q, summed as doubles and reduced every 8 digits
//     (below 2^45 throughout);
//   integer: Montgomery products, two 32-bit steps.  With T = d k for a digit
//     d < 16 q < 2^64 and a canonical key entry k, T < 2^124, each step adds
//     the multiple m q that clears the lowest word and drops it: T / 2^64
//     (mod q) below 2q.  Four of them and a reduced sum stay below 11 q; the
//     factor 2^64 comes back with the last reduction, one product by 2^64 mod
//     q.  (128-bit sums need no reduction per product but twice the registers,
//     which then spill.)
struct SumFp {
    static constexpr int kIn = 1;  // bound of total()
    double q, qinv;
    typedef double S;
    CK_HD void mac(S &s, u64 y, u64 w) const {
        s += fp_mulmod_q(u64_as_f64(y), small_to_f64(w), q, qinv);
    }
    CK_HD static bool full(u32 j) { return (j & 7) == 7; }
    CK_HD S reduced(S s) const { return fp_reduce(s, q, qinv); }
    CK_HD u64 total(S s) const { return f64_as_u64(fp_reduce(s, q, qinv)); }
};
struct SumInt {
    static constexpr int kIn = 3;
    u64 q, r_hi, r_lo;  // modulus, floor(2^128 / q)
    u32 qi;             // -q^-1 mod 2^32
    typedef u64 S;
    CK_HD SumInt(u64 q_, u64 hi, u64 lo) : q(q_), r_hi(hi), r_lo(lo) {
        u32 x = (u32)q;  // q q == 1 mod 8; each step doubles the correct bits
#pragma unroll
        for (int it = 0; it < 4; ++it) x *= 2u - (u32)q * x;
        qi = 0u - x;
    }
    CK_HD void mac(S &s, u64 y, u64 w) const {
        const u32 q0 = (u32)q, q1 = (u32)(q >> 32);
        const unsigned __int128 T = (unsigned __int128)y * w;
        const u32 m0 = (u32)T * qi;
        const u64 c0 = (u64)m0 * q1 + (((u64)m0 * q0 + (u32)T) >> 32);
        const unsigned __int128 U = (T >> 32) + c0;  // three words
        const u32 m1 = (u32)U * qi;
        const u64 c1 = (u64)m1 * q1 + (((u64)m1 * q0 + (u32)U) >> 32);
        s += (u64)(U >> 32) + c1;
    }
    CK_HD static bool full(u32 j) { return (j & 3) == 3; }
    CK_HD S reduced(S s) const { return shoup_lazy3(s, 1, r_hi, q); }
    CK_HD u64 total(S s) const { return shoup_lazy3(s, 0 - r_hi * q, r_lo, q); }
};

}  // namespace ck
