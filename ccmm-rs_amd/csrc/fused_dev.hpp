// Device helpers of the fused passes (fused.hip) and of the lifts in keyswitch.hip.
#pragma once
#include "fused.hpp"
#include "row_sums.hpp"

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

// Input of limb prime P, largest bounds after it (see RowFp, RowInt):
//   plain: canonical residues;
//   residue: canonical modulo another prime of the plan (`limit`);
//   digit: a balanced digit, |d| <= limit <= 2^62.
// FP64 limbs take values up to 2^44 whole (with eight stages of 0.52 q they
// stay below 2^45) and cut larger ones at bit 30; integer limbs take residues
// up to 4q whole, add q to negative digits when limit < q, and reduce the rest
// (below 2^64) into 3q.  Which of them is the same for a whole block.
//   bytes: |d| <= 128, below every prime of a two-pass degree;
//   block: a mixed-radix value, see col_blocks; within 0.54 q or below 2q.
constexpr int kColFpIn = 16, kColIntIn = 4;
constexpr u64 kColFpWhole = 1ull << 44;

template <int M>
__device__ __forceinline__ void col_lift(u64 (&v)[M], u32 kind, u64 limit, const RowFp &ar, const CK_CONST_AS DevPrime &) {
    if (kind == kColPlain || limit <= kColFpWhole) {  // limit 0 for bytes
#pragma unroll
        for (int i = 0; i < M; ++i) v[i] = f64_as_u64(signed_to_f64(v[i]));
        return;
    }
    const double k30 = fp_reduce(1073741824.0, ar.q, ar.qinv);
#pragma unroll
    for (int i = 0; i < M; ++i) {
        const double hi = signed_to_f64((u64)((int64_t)v[i] >> 30)), lo = (double)(u32)(v[i] & 0x3fffffffu);
        v[i] = f64_as_u64(lo + fp_mulmod_q(hi, k30, ar.q, ar.qinv));
        if ((i & 3) == 3) sched_fence();
    }
}
template <int M>
__device__ __forceinline__ void col_lift(u64 (&v)[M], u32 kind, u64 limit, const RowInt &ar, const CK_CONST_AS DevPrime &P) {
    if (kind == kColInt8 || (kind == kColDigit && limit < ar.q)) {
#pragma unroll
        for (int i = 0; i < M; ++i) v[i] += (int64_t)v[i] < 0 ? ar.q : 0;
    } else if (kind == kColDigit || (kind == kColResidue && limit > 4 * ar.q)) {
        // a multiple of q from limit to limit + 2q makes every digit positive
        const u64 up = kind == kColDigit ? (mulhi64(limit, P.br_hi) + 2) * ar.q : 0;
#pragma unroll
        for (int i = 0; i < M; ++i) {
            v[i] = shoup_lazy3(v[i] + up, 1, P.br_hi, ar.q);
            if ((i & 3) == 3) sched_fence();
        }
    }
}

// a canonical residue as a product's first operand
__device__ __forceinline__ u64 sum_input(u64 x, const RowFp &) { return f64_as_u64(small_to_f64(x)); }
__device__ __forceinline__ u64 sum_input(u64 x, const RowInt &) { return x; }

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
