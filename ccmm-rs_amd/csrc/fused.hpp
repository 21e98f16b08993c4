// Interface of the fused NTT passes (fused.hip).
#pragma once
#include "internal.hpp"

namespace ck {

// The passes serve two-pass degrees with primes below 2^60 (RowInt's lazy range): column passes
// that read a key switch's digits in the form it has them, and row passes
// that do the pointwise work between the forward and the inverse transform.
bool fused_rows_apply(const ckks_rns_plan *plan);
// Row products psi^((2u+1) t) of one prime's table into out (FP64 primes:
// doubles, others: Tw), queued on s.
int build_row_products(hipStream_t s, const Tw *table, u64 q, bool fp, u32 logn, void *out);

// Input of a forward column pass.
enum ColKind {
    kColPlain = 0,    // polynomials [p][limb][N], canonical residues
    kColResidue = 1,  // digit j of a ciphertext is its limb j ([ct][digits][N]), lifted to every limb
    kColDigit = 2,    // balanced digits, int64 [ct][digits][N], |d| <= limit, lifted to every limb
    kColBlock = 3,    // digit j is given by its mixed-radix digits ([ct][.][N], see ColBlock)
    kColInt8 = 4,     // signed bytes [p][N], the same in every limb
};
// What the inverse column pass adds to its result v on the way out.
enum ColAdd {
    kAddNone = 0,
    kAddMessage = 1,  // m + e - v: m like the output, e int64 [p][N]
    kAddBody = 2,     // m + v
};
// A gadget block as kColBlock evaluates it: the block's value is sum_t c_t W_t,
// c_t < 2^41 the mixed-radix digits (limbs first .. of the ciphertext's data);
// split: digit 0 is below 2^60 and enters as its low 30 bits (t = 0) and the
// rest (t = 1, weight 2^30 W_0).  Row i of `rows` holds, per term, W_t mod q_i
// and fl(that / q_i) as double bits.
constexpr int kColTerms = 13;
struct ColBlock {
    u32 first, terms, split;
    const u64 *rows;  // [limb][kColTerms][2]
};
// Forward: `in` (as kind says, `stride` elements between polynomials, lifts:
// between ciphertexts) to inter-pass data in `out`.  Inverse: inter-pass data
// `in` to polynomials in `out`, `stride` apart.  Inter-pass data is limb-major
// ([limb][poly][N]), already multiplied (forward), not yet multiplied
// (inverse) by the row products.
struct ColCall {
    const ckks_rns_plan *plan;
    const u64 *in;
    u64 *out;
    size_t n_polys, n_limbs, stride;
    int kind = kColPlain;
    size_t digits = 1;  // polynomials per ciphertext (lifts)
    u64 limit = 0;      // kColDigit
    const ColBlock *blocks = nullptr;  // kColBlock: one per digit, device memory
    int add = kAddNone;                // inverse
    const u64 *m = nullptr;
    size_t m_stride = 0;
    const int64_t *e = nullptr;
};
int launch_columns(ckks_context *ctx, const ColCall *calls, size_t count, bool forward);

// Key inner products between the column passes of key switches by up to
// kRowJobs keys of one shape: the forward row pass of the digits, the products
// with the key and the inverse row pass of both sums.
constexpr size_t kRowJobs = 16;
struct RowMacJob {
    const u64 *digits;   // inter-pass, polynomials [ct][j]
    const u64 *kb, *ka;  // [dnum][limbs][N], NTT domain, natural order
    u64 *out;            // inter-pass, polynomials [ct][2]
    u32 n_cts, first;    // first: set by the launch
};
struct RowMac {
    const ckks_rns_plan *plan;
    size_t dnum, limbs;
    bool xcd_order;  // ciphertexts of one key tile on one XCD
    size_t count;
    RowMacJob e[kRowJobs];
};
int launch_row_mac(ckks_context *ctx, RowMac &m);

// Products between the column passes, in place of the first operand's
// inter-pass data (n_polys polynomials of `limbs` limbs).
struct RowMul {
    const ckks_rns_plan *plan;
    u64 *x;
    size_t n_polys, limbs;
    // the other operand: inter-pass data of one polynomial for all of them, or
    const u64 *y = nullptr;
    // NTT-domain values in natural order, [limb][N] for every `share`
    // polynomials, w_stride apart
    const u64 *w = nullptr;
    size_t share = 1, w_stride = 0;
};
int launch_row_mul(ckks_context *ctx, const RowMul &m);

// Tensor of ciphertext pairs: inter-pass b0, a0, b1, a1 (n_cts polynomials
// each) to inter-pass b0 b1, b0 a1 + a0 b1, a0 a1 in the place of b0, a0, b1.
int launch_row_tensor(ckks_context *ctx, const ckks_rns_plan *plan, u64 *const x[4], size_t n_cts, size_t limbs);

// Hoisted rotations of one batch of digits by several exponents: for each, the
// products with its key (entries permuted by k^-1), the corrections, sigma_k
// and the inverse row pass of both sums.
constexpr int kRowRotations = 16;
struct RowRotation {
    const u64 *kb, *ka;  // [dnum][limbs][N], NTT domain, natural order
    const u64 *tb, *ta;  // [limbs][N] added to the sums, or null
    u64 *out;            // inter-pass, polynomials [ct][2]
    u32 kinv;            // k^-1 modulo 2N
};
struct RowRotate {
    const ckks_rns_plan *plan;
    const u64 *digits;  // [ct][dnum][limbs][N], NTT domain
    const u64 *bhat;    // added to every first sum on limbs below q_limbs, [ct][q_limbs][N], or null
    size_t n_cts, dnum, limbs, q_limbs;
    const RowRotation *e;
    size_t count;
};
int launch_row_rotate(ckks_context *ctx, const RowRotate &r);

// Single-pass degrees (N <= 4096, every plan prime < 2^60; small.hip).
bool small_tiles_apply(const ckks_rns_plan *plan);
constexpr size_t kSmallJobs = 16;
struct SmallCall {
    const ckks_rns_plan *plan;
    const u64 *in;
    u64 *out;
    size_t n_polys, n_limbs, in_stride, out_stride;
    // nonzero: forward, the polynomials are the single-limb gadget digits of
    // n_polys / digits ciphertexts (in_stride apart, sigma_k of them for kinv
    // nonzero); inverse, they are the two key products of n_polys / 2
    // ciphertexts' transformed digits [ct][digit][limb][N]
    size_t digits = 0;
    u64 kinv = 0;
    const u64 *kb = nullptr, *ka = nullptr;
};
int launch_small(ckks_context *ctx, const SmallCall *calls, size_t count, bool forward);

// out[e] = sum_t ct[t] pt[e][t] over NTT-domain ciphertexts [2][limbs][N] and
// plaintexts [limbs][N]; plans of primes below 2^60.
constexpr size_t kMacPointers = 384;
bool mac_tiles_apply(const ckks_rns_plan *plan);
int launch_mac_lists(const ckks_rns_plan *plan, const u64 *const *cts, const u64 *const *pts, size_t count,
                     u64 *const *outs, size_t n_outs, size_t n_limbs);

}  // namespace ck
