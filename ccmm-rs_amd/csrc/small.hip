// Single-pass transforms (N <= 4096) and the key switch built on them: see
// small_tile.hpp.  Against 256 threads of sixteen residues, separate lifts and
// products, at N = 2^12 (a 60-bit and three 40-bit primes): 2 polynomials
// 12.3 -> 8.8 us (the workgroup's latency), 4096 polynomials 368 -> 352 us
// forward, 418 -> 359 us inverse (HBM: 4.3 GB at 4.79 TB/s is 224 us);
// single-limb rotation of one ciphertext 43.5 -> 30.7 us, of 1024 2.51 -> 0.94 ms.
#include "fused_dev.hpp"
#include "small_tile.hpp"

namespace ck {

bool small_tiles_apply(const ckks_rns_plan *plan) {
    if (plan->logn < 10 || plan->logn > 12) return false;
    for (u64 q : plan->moduli)
        if (q >= kLazyModulusBound) return false;
    return true;
}

struct SmallEntry {
    const u64 *src;
    u64 *dst;
    u64 src_stride, dst_stride;  // between polynomials (digits: ciphertexts of src)
    const DevPrime *primes;
    u64 kinv;                    // digits: the source is sigma_k's
    const u64 *kb, *ka;          // products: [dnum][limbs][N]
    u32 n_polys, n_limbs, digits, first;
};

struct SmallLaunch {
    SmallEntry e[kSmallJobs];
    u32 count;
};

// Forward transform of canonical residues, or of single-limb gadget digits:
// polynomial p is the residues of limb p mod `digits` of ciphertext
// p / digits, lifted to the target limb.
template <int L, bool DIGITS, class Ar>
__device__ __forceinline__ void small_forward(const SmallEntry &e, const CK_CONST_AS DevPrime &P, const Ar &ar,
                                              u32 limb, u32 poly, u64 (*lds)[SmallTile<L>::LDS]) {
    typedef SmallTile<L> S;
    const u32 tid = threadIdx.x;
    const u64 N = (u64)1 << L;
    u64 v[8];
    int b[8];
    if constexpr (DIGITS) {
        const u32 j = poly % e.digits, mask2 = (2u << L) - 1;
        const u64 qj = const_table(e.primes)[j].q;
        const u64 *src = e.src + poly / e.digits * e.src_stride + j * N;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const u32 n = tid + i * S::THREADS;
            u32 from = n;
            bool neg = false;
            if (e.kinv) {
                from = (n * (u32)e.kinv) & mask2;
                neg = from >= (u32)N;
                from &= (u32)N - 1;
            }
            v[i] = load_at(src, from * 8);
            if (neg) v[i] = neg_mod(v[i], qj);
        }
        col_lift(v, kColResidue, qj, ar, P);
        S::set(b, Ar::kFp ? kColFpIn : kColIntIn);
    } else {
        const u64 *src = e.src + poly * e.src_stride + limb * N;
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = load_at(src + i * S::THREADS, tid * 8);
        if constexpr (Ar::kFp) {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = f64_as_u64(small_to_f64(v[i]));
        }
        S::set(b, Ar::kFp ? 2 : 1);
    }
    const typename S::Tws wa = S::template twiddles<0>(P.fwd, tid), wb = S::template twiddles<1>(P.fwd, tid),
                          wc = S::template twiddles<2>(P.fwd, tid), wd = S::template twiddles<3>(P.fwd, tid);
    S::template fwd<0>(v, b, wa, ar);
    S::template put<0>(v, tid, lds[0]);
    __syncthreads();
    S::template get<1>(v, tid, lds[0]);
    S::level(b);
    S::template fwd<1>(v, b, wb, ar);
    S::template put<1>(v, tid, lds[1]);
    __syncthreads();
    S::template get<2>(v, tid, lds[1]);
    S::level(b);
    S::template fwd<2>(v, b, wc, ar);
    S::template put<2>(v, tid, lds[0]);
    __syncthreads();
    S::template get<3>(v, tid, lds[0]);
    S::level(b);
    S::template fwd<3>(v, b, wd, ar);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        if constexpr (Ar::kFp) v[i] = fp_residue(u64_as_f64(v[i]), ar.q, ar.qinv);
        else ar.reduce_to(v[i], b[i], 1);
    }
    S::template put<3>(v, tid, lds[1]);
    __syncthreads();
    S::get_natural(v, tid, lds[1]);
    u64 *dst = e.dst + poly * e.dst_stride + limb * N;
#pragma unroll
    for (int i = 0; i < 8; ++i) *(u64 *)((char *)(dst + i * S::THREADS) + tid * 8) = v[i];
}

// Inverse transform of canonical residues, or of the key products of a
// ciphertext's digits: polynomial p is component p mod 2 of ciphertext p / 2.
template <int L, bool MAC, class Ar, class Sum>
__device__ __forceinline__ void small_inverse(const SmallEntry &e, const CK_CONST_AS DevPrime &P, const Ar &ar,
                                              const Sum &sum, u32 limb, u32 poly, u64 (*lds)[SmallTile<L>::LDS]) {
    typedef SmallTile<L> S;
    const u32 tid = threadIdx.x;
    const u64 N = (u64)1 << L;
    u64 v[8];
    int b[8];
    const typename S::Tws wd = S::template twiddles<3>(P.inv, tid);
    if constexpr (MAC) {
        const u64 stride = (u64)e.n_limbs * N;
        const u64 *d = e.src + (u64)(poly / 2) * e.digits * stride + limb * N;
        const u64 *k = (poly & 1 ? e.ka : e.kb) + limb * N;
        typename Sum::S s[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) s[i] = 0;
        u64 x[8], w[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            x[i] = load_at(d + i * S::THREADS, tid * 8);
            w[i] = load_at(k + i * S::THREADS, tid * 8);
        }
#pragma unroll 1
        for (u32 j = 0;; ++j) {
            u64 nx[8], nw[8];
            const bool last = j + 1 == e.digits;
            d += stride;
            k += stride;
            if (!last) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    nx[i] = load_at(d + i * S::THREADS, tid * 8);
                    nw[i] = load_at(k + i * S::THREADS, tid * 8);
                }
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) sum.mac(s[i], sum_input(x[i], ar), w[i]);
            if (last) break;
            if (Sum::full(j)) {
#pragma unroll
                for (int i = 0; i < 8; ++i) s[i] = sum.reduced(s[i]);
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                x[i] = nx[i];
                w[i] = nw[i];
            }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = sum.total(s[i]);
        S::set(b, Sum::kIn);
    } else {
        const u64 *src = e.src + poly * e.src_stride + limb * N;
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = sum_input(load_at(src + i * S::THREADS, tid * 8), ar);
        S::set(b, Ar::kFp ? 2 : 1);
    }
    S::put_natural(v, tid, lds[0]);
    const typename S::Tws wc = S::template twiddles<2>(P.inv, tid), wb = S::template twiddles<1>(P.inv, tid),
                          wa = S::template twiddles<0>(P.inv, tid);
    __syncthreads();
    S::template get<3>(v, tid, lds[0]);
    S::template inv<3>(v, b, wd, ar);
    S::template put<3>(v, tid, lds[1]);
    __syncthreads();
    S::template get<2>(v, tid, lds[1]);
    S::level(b);
    S::template inv<2>(v, b, wc, ar);
    S::template put<2>(v, tid, lds[0]);
    __syncthreads();
    S::template get<1>(v, tid, lds[0]);
    S::level(b);
    S::template inv<1>(v, b, wb, ar);
    S::template put<1>(v, tid, lds[1]);
    __syncthreads();
    S::template get<0>(v, tid, lds[1]);
    S::level(b);
    S::template inv<0>(v, b, wa, ar);
    u64 *dst = e.dst + poly * e.dst_stride + limb * N;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        u64 r;
        if constexpr (Ar::kFp)
            r = fp_residue(fp_mulmod(u64_as_f64(v[i]), P.ninv_d, P.ninv_p, ar.q), ar.q, ar.qinv);
        else
            r = shoup(v[i], P.ninv, P.ninv_q, ar.q);
        *(u64 *)((char *)(dst + i * S::THREADS) + tid * 8) = r;
    }
}

// EXTRA: gadget digits (forward) or key products (inverse) as input
template <int L, bool FWD, bool EXTRA>
__global__ __launch_bounds__(512, 4) void k_small(SmallLaunch l) {
    __shared__ u64 lds[2][SmallTile<L>::LDS];
    u32 i = 0;
    while (i + 1 < l.count && blockIdx.x >= l.e[i + 1].first) ++i;
    const SmallEntry &e = l.e[i];
    const u32 x = blockIdx.x - e.first, limb = x % e.n_limbs, poly = x / e.n_limbs;
    const CK_CONST_AS DevPrime &P = const_table(e.primes)[limb];
    const RowFp fp{P.qd, P.qinv};
    const RowInt in{P.q};
    if constexpr (FWD) {
        if (P.fp) small_forward<L, EXTRA>(e, P, fp, limb, poly, lds);
        else small_forward<L, EXTRA>(e, P, in, limb, poly, lds);
    } else {
        if (P.fp) small_inverse<L, EXTRA>(e, P, fp, SumFp{P.qd, P.qinv}, limb, poly, lds);
        else small_inverse<L, EXTRA>(e, P, in, SumInt(P.q, P.br_hi, P.br_lo), limb, poly, lds);
    }
}

int launch_small(ckks_context *ctx, const SmallCall *calls, size_t count, bool forward) {
    for (u32 logn = 10; logn <= 12; ++logn)
        for (int extra = 0; extra < 2; ++extra) {
            SmallLaunch l{};
            size_t blocks = 0;
            for (size_t i = 0; i < count; ++i) {
                const SmallCall &c = calls[i];
                if (c.n_polys == 0 || c.plan->logn != logn || (c.digits != 0) != (extra != 0)) continue;
                if (!small_tiles_apply(c.plan) || l.count == kSmallJobs)
                    return fail(CKKS_ERR_UNSUPPORTED, "single-pass tiles: N <= 4096, primes below 2^60, 16 entries");
                l.e[l.count++] = SmallEntry{c.in, c.out, c.in_stride, c.out_stride, c.plan->d_primes, c.kinv, c.kb, c.ka,
                                            (u32)c.n_polys, (u32)c.n_limbs, (u32)c.digits, (u32)blocks};
                blocks += c.n_polys * c.n_limbs;
            }
            if (blocks == 0) continue;
            if (blocks >= (1ull << 31)) return fail(CKKS_ERR_INVALID, "NTT batch too large for one launch");
            const dim3 g((u32)blocks), t(1u << (logn - 3));
            switch (logn * 4 + (forward ? 2 : 0) + extra) {
#define CK_SM(L)                                                                                              \
    case L * 4: hipLaunchKernelGGL((k_small<L, false, false>), g, t, 0, ctx->stream, l); break;               \
    case L * 4 + 1: hipLaunchKernelGGL((k_small<L, false, true>), g, t, 0, ctx->stream, l); break;            \
    case L * 4 + 2: hipLaunchKernelGGL((k_small<L, true, false>), g, t, 0, ctx->stream, l); break;            \
    case L * 4 + 3: hipLaunchKernelGGL((k_small<L, true, true>), g, t, 0, ctx->stream, l); break;
                CK_SM(10) CK_SM(11) CK_SM(12)
#undef CK_SM
            }
            CK_HIP(hipGetLastError());
        }
    return CKKS_OK;
}

}  // namespace ck
