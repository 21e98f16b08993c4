// Plaintext-diagonal inner sums over NTT-resident ciphertexts, several sums of
// the same ciphertexts at a time.
//
// The sums stream their plaintexts (every one is read once) and the
// ciphertexts, which all of them share: a launch per sum reads count * 2 polynomials
// of ciphertexts for count of plaintexts.  Eight sums share each ciphertext
// entry in registers (two components: 16 running sums a thread), and a
// plaintext entry serves both components.  FP64 products for FP64 limbs,
// Montgomery sums for the others, in place of a 128-bit Barrett product each.
// 16 sums of 16 terms at N = 2^14, 8 limbs (268 MB of plaintexts): 66 us in
// one call, 240 us as 16 launches of one.
#include "fused_dev.hpp"

namespace ck {

bool mac_tiles_apply(const ckks_rns_plan *plan) {
    for (u64 q : plan->moduli)
        if (q >= kLazyModulusBound) return false;
    return true;
}

constexpr size_t kMacOuts = 16;

struct MacLists {
    const u64 *p[kMacPointers];  // count ciphertexts, then count plaintexts of every output
    u64 *out[kMacOuts];
    const DevPrime *primes;
    u32 count, n_outs, n_limbs, logn;
};

template <int E, class Ar, class Sum>
__device__ __forceinline__ void mac_thread(const MacLists &a, const Ar &ar, const Sum &sum, u32 limb, u64 n, u32 e0) {
    const u64 N = (u64)1 << a.logn, comp = (u64)a.n_limbs * N, off = (u64)limb * N + n;
    typename Sum::S s[E][2];
#pragma unroll
    for (int e = 0; e < E; ++e) s[e][0] = s[e][1] = 0;
#pragma unroll 1
    for (u32 t = 0; t < a.count; ++t) {
        const u64 *ct = a.p[t] + off;
        const u64 x = sum_input(ct[0], ar), y = sum_input(ct[comp], ar);
        u64 w[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const u32 o = e0 + e < a.n_outs ? e0 + e : e0;  // past the last: not stored
            w[e] = ld_stream(a.p[(o + 1) * a.count + t] + off);
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
            sum.mac(s[e][0], x, w[e]);
            sum.mac(s[e][1], y, w[e]);
        }
        if (Sum::full(t)) {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                s[e][0] = sum.reduced(s[e][0]);
                s[e][1] = sum.reduced(s[e][1]);
            }
        }
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
        if (e0 + e >= a.n_outs) break;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            u64 r;
            if constexpr (Ar::kFp) {
                r = fp_residue(s[e][c], ar.q, ar.qinv);
            } else {
                r = sum.total(s[e][c]);
                int b = Sum::kIn;
                ar.reduce_to(r, b, 1);
            }
            a.out[e0 + e][c * comp + off] = r;
        }
    }
}

template <int E>
__global__ __launch_bounds__(256) void k_mac_lists(MacLists a) {
    const u32 chunks = 1u << (a.logn - 8);
    const u32 chunk = blockIdx.x % chunks, r = blockIdx.x / chunks, limb = r % a.n_limbs, e0 = r / a.n_limbs * E;
    const u64 n = (u64)chunk * 256 + threadIdx.x;
    const CK_CONST_AS DevPrime &P = const_table(a.primes)[limb];
    if (P.fp)
        mac_thread<E>(a, RowFp{P.qd, P.qinv}, SumFp{P.qd, P.qinv}, limb, n, e0);
    else
        mac_thread<E>(a, RowInt{P.q}, SumInt(P.q, P.br_hi, P.br_lo), limb, n, e0);
}

int launch_mac_lists(const ckks_rns_plan *plan, const u64 *const *cts, const u64 *const *pts, size_t count,
                     u64 *const *outs, size_t n_outs, size_t n_limbs) {
    if (!mac_tiles_apply(plan)) return fail(CKKS_ERR_UNSUPPORTED, "shared inner sums: primes below 2^60");
    if (count == 0 || n_outs == 0 || n_outs > kMacOuts || count * (n_outs + 1) > kMacPointers)
        return fail(CKKS_ERR_INVALID, "shared inner sums: at most 16, 384 operands");
    MacLists a{};
    for (size_t t = 0; t < count; ++t) a.p[t] = cts[t];
    for (size_t t = 0; t < n_outs * count; ++t) a.p[count + t] = pts[t];
    for (size_t e = 0; e < n_outs; ++e) a.out[e] = outs[e];
    a.primes = plan->d_primes;
    a.count = (u32)count;
    a.n_outs = (u32)n_outs;
    a.n_limbs = (u32)n_limbs;
    a.logn = plan->logn;
    const u32 E = n_outs == 1 ? 1 : n_outs <= 4 ? 4 : 8;
    const dim3 g((u32)(((n_outs + E - 1) / E * n_limbs) << (plan->logn - 8))), t(256);
    hipStream_t s = plan->ctx->stream;
    if (E == 1) hipLaunchKernelGGL(k_mac_lists<1>, g, t, 0, s, a);
    else if (E == 4) hipLaunchKernelGGL(k_mac_lists<4>, g, t, 0, s, a);
    else hipLaunchKernelGGL(k_mac_lists<8>, g, t, 0, s, a);
    CK_HIP(hipGetLastError());
    return CKKS_OK;
}

}  // namespace ck
