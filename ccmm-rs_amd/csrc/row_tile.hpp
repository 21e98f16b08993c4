// Row-pass tile of the fused kernels: forward row pass, a pointwise product
// in the NTT domain and the inverse row pass without leaving the workgroup.
//
// The row pass of a two-pass transform (ntt_tile.hpp) works on rows of N2 =
// 2^L residues; row m = bitrev(u) holds a polynomial modulo X^N2 - rho^N2,
// rho = psi^(2u+1).  Substituting X -> rho X turns every row into the same
// cyclic transform modulo X^N2 - 1, so
//   forward: element t times Z[m N2 + t] = psi^((2u+1) t) (the column pass
//            does it on its way out), then cyclic CT stages whose twiddle at
//            stage s, block j = t >> (L-s) is T[j];
//   inverse: cyclic GS stages with Tinv[j], then times Zi = psi^-((2u+1) t)
//            (the column pass does it on its way in).
// T is the column pass's table (T[k] = psi^bitrev(k) depends on the bits of k
// only through psi^(N phi(k)), phi the bit-reversed fraction, so its first
// 2^(L-1) entries are the cyclic twiddles of every row).  Against per-row
// twiddles this takes one product per residue for the row and leaves j = 0
// butterflies without a product: per 8 residues of an FP64 row 25 products
// (and 8 in the column pass) and no twiddle arithmetic where the row-factored
// twiddles take 32 products plus one more per distinct twiddle.  The twiddles of the first six stages
// are uniform over a wave (geometries below) and come through the scalar unit.
//
// A tile is 4096 residues (TB = 12): 2^L residues of 2^(12-L) rows, 8 per thread
// in 512 threads, three rounds of at most 3 stages with an LDS exchange between
// rounds.  TB = 11 halves rows and threads (round B's twiddles are then uniform
// over half a wave only) for launches of few tiles.  Eight residues a thread (not 16) leave the registers for two
// accumulators per residue.
#pragma once
#include "ntt_tile.hpp"

namespace ck {

// y w mod q (exact, |r| < 0.52 q) for integer-valued doubles, |y| < 2^45,
// 0 <= w < q < 2^41, without a precomputed w / q: the quotient estimate
// fl(fl(y w) fl(1/q)) carries three roundings, |error| < 3 2^-53 2^45 < 2^-6.
CK_HD double fp_mulmod_q(double y, double w, double q, double qinv) {
#pragma clang fp contract(off)
    const double hi = y * w;
    const double lo = __builtin_fma(y, w, -hi);
    const double k = __builtin_rint(hi * qinv);
    return __builtin_fma(-k, q, hi) + lo;
}

// Primes of the integer arithmetic below: q < 2^60, so 16 q fits 64 bits and
// butterflies need a conditional subtraction only where the bound tracked
// per residue (in units of q) would pass 16.
constexpr u64 kLazyModulusBound = 1ull << 60;

// y w - h q in [0, 3q) with h = floor(y wq / 2^64) or one less: the product of
// the low words of y and wq, which only adds a carry, is left out.
CK_HD u64 shoup_lazy3(u64 y, u64 w, u64 wq, u64 q) {
    const u32 y0 = (u32)y, y1 = (u32)(y >> 32), a0 = (u32)wq, a1 = (u32)(wq >> 32);
    const u64 m1 = (u64)y0 * a1;
    const u64 m2 = (u64)y1 * a0 + (u32)m1;
    const u64 h = (u64)y1 * a1 + (m1 >> 32) + (m2 >> 32);
    return y * w - h * q;
}

// Arithmetic of one limb, with the compile-time bound of every residue kept
// beside it (int references that fold away once the rounds are unrolled).
struct RowFp {
    typedef double V;
    static constexpr bool kFp = true;
    static constexpr int kMax = 30;   // bounds in units of 0.52 q: |y| < 2^45 = 16 q, fp_mulmod's range
    double q, qinv;
    CK_HD static V from_bits(u64 x) { return u64_as_f64(x); }
    CK_HD static u64 to_bits(V x) { return f64_as_u64(x); }
    // the table's w / q is not read: a register pair less per twiddle
    CK_HD V mul(V y, const Tw &w) const { return fp_mulmod_q(y, u64_as_f64(w.w), q, qinv); }
    CK_HD void reduce(V &x, int &b) const {
        x = fp_reduce(x, q, qinv);
        b = 1;
    }
    CK_HD void fit(V &x, V &y, int &bx, int &by) const {
        if (bx + by > kMax) reduce(x, bx);
        if (bx + by > kMax) reduce(y, by);
    }
    CK_HD void settle(V &x, int &b) const {
        if (b > 3) reduce(x, b);
    }
    // times a row product
    typedef double Z;
    static constexpr int kZ = 1;  // bound after it
    CK_HD u64 times(u64 x, Z z) const { return f64_as_u64(fp_mulmod_q(u64_as_f64(x), z, q, qinv)); }
    CK_HD void ct(V &x, V &y, const Tw &w, int &bx, int &by) const {
        if (bx + 1 > kMax) reduce(x, bx);
        const V a = x, t = mul(y, w);
        x = a + t;
        y = a - t;
        bx = by = bx + 1;
    }
    CK_HD void ct1(V &x, V &y, int &bx, int &by) const {
        fit(x, y, bx, by);
        const V a = x, b = y;
        x = a + b;
        y = a - b;
        bx = by = bx + by;
    }
    CK_HD void gs(V &x, V &y, const Tw &w, int &bx, int &by) const {
        fit(x, y, bx, by);
        const V a = x, b = y;
        x = a + b;
        y = mul(a - b, w);
        bx += by;
        by = 1;
    }
    CK_HD void gs1(V &x, V &y, int &bx, int &by) const { ct1(x, y, bx, by); }
};

struct RowInt {
    typedef u64 V;
    static constexpr bool kFp = false;
    static constexpr int kMax = 16;  // bounds in units of q < 2^60
    u64 q;
    // k q kept out of the compiler's sight: it would fold k q + x into two
    // 64-bit multiply-adds where a uniform k q takes one addition
    CK_HD u64 times_q(int k) const {
        u64 m = q * (u64)k;
#if defined(__HIP_DEVICE_COMPILE__)
        asm("" : "+s"(m));
#endif
        return m;
    }
    CK_HD static V from_bits(u64 x) { return x; }
    CK_HD static u64 to_bits(V x) { return x; }
    CK_HD V mul(V y, const Tw &w) const { return shoup_lazy3(y, w.w, w.wq, q); }
    // below b q -> below target q by conditional subtractions of 8q, 4q, ..
    CK_HD void reduce_to(V &x, int &b, int target) const {
#pragma unroll
        for (int s = 8; s >= 1; s >>= 1)
            if (b > target && b > s) {
                const u64 sq = times_q(s);
                x = x >= sq ? x - sq : x;
                b = b - s > s ? b - s : s;
            }
    }
    CK_HD void fit(V &x, V &y, int &bx, int &by) const {
        if (bx + by > kMax) reduce_to(x, bx, 8);
        if (bx + by > kMax) reduce_to(y, by, 8);
    }
    CK_HD void settle(V &x, int &b) const { reduce_to(x, b, 4); }
    typedef Tw Z;
    static constexpr int kZ = 3;
    CK_HD u64 times(u64 x, const Z &z) const { return shoup_lazy3(x, z.w, z.wq, q); }
    CK_HD void ct(V &x, V &y, const Tw &w, int &bx, int &by) const {
        if (bx + 3 > kMax) reduce_to(x, bx, 8);
        const V a = x, t = mul(y, w);
        x = a + t;
        y = a + times_q(3) - t;
        bx = by = bx + 3;
    }
    CK_HD void ct1(V &x, V &y, int &bx, int &by) const {
        fit(x, y, bx, by);
        const V a = x, b = y;
        x = a + b;
        y = a + times_q(by) - b;
        bx = by = bx + by;
    }
    CK_HD void gs(V &x, V &y, const Tw &w, int &bx, int &by) const {
        fit(x, y, bx, by);
        const V a = x, b = y;
        x = a + b;
        y = mul(a + times_q(by) - b, w);
        bx += by;
        by = 3;
    }
    CK_HD void gs1(V &x, V &y, int &bx, int &by) const { ct1(x, y, bx, by); }
};

// Ends a scheduling region: keeps the compiler from issuing the twiddle loads
// and products of many butterflies at once, which costs registers.
CK_HD void sched_fence() {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_sched_barrier(0);
#endif
}

// LDS placement of the column tile: linear address (t << CL) | col with bits
// 0..4 XORed by kRowSwizzle[k] for every set bit 5 + k: no padding, so five
// 32 KiB tiles fit a CU.  The seven columns were searched so that in every
// geometry the six lane bits of a wave, and its first five, map onto five
// independent low bits: 64 lanes of 8 bytes touch each 8-byte slot twice.
constexpr u32 kRowSwizzle[7] = {31, 17, 26, 22, 5, 21, 30};

CK_HD u32 row_swizzle(u32 a) {
    u32 x = a;
#pragma unroll
    for (int k = 0; k < 7; ++k)
        if ((a >> (5 + k)) & 1u) x ^= kRowSwizzle[k];
    return x;
}

// Geometry A holds the top three bits of t in a thread's registers (lanes
// walk t: rows are read and written in 2^(L-3)-residue runs), B the next
// three (lanes: the rest of t below, then columns; the wave number is the top
// of t, so the twiddles of stages 3..5 are wave-uniform), C the low L - 6
// bits of t and the low 9 - L columns (lanes walk columns, so the natural
// positions bitrev(t) N1 + u of a wave are whole 128-byte runs).
// two adjacent residues, 16-byte aligned in LDS
struct alignas(16) Pair {
    u64 x, y;
};

template <int L, int TB = 12>
struct RowTile {
    static constexpr int CL = TB - L, KC = L - 6, EX = 3 - KC;
    static constexpr u32 THREADS = 1u << (TB - 3);
    static_assert(L >= 7 && L <= 9 && CL >= 2 && CL >= EX, "rows of 128 .. 512 residues");

    CK_HD static u32 t_of(int geo, u32 tid, int i) {
        if (geo == 0) return (tid & ((1u << (L - 3)) - 1)) | ((u32)i << (L - 3));
        if (geo == 1) return (tid & ((1u << KC) - 1)) | ((u32)i << KC) | ((tid >> (KC + CL)) << (KC + 3));
        return ((tid >> (CL - EX)) << KC) | ((u32)i >> EX);
    }
    CK_HD static u32 col_of(int geo, u32 tid, int i) {
        if (geo == 0) return tid >> (L - 3);
        if (geo == 1) return (tid & ((1u << (KC + CL)) - 1)) >> KC;
        return ((tid & ((1u << (CL - EX)) - 1)) << EX) | ((u32)i & ((1u << EX) - 1));
    }
    // LDS placement: slot a + 2 (a >> 4) of linear address a = (t << CL) | col.
    // Additive over disjoint bits, so register i is the thread's address plus
    // a constant the instruction carries as its offset; 64 lanes of 8 bytes
    // touch an 8-byte slot two to four times (two is the least), geometry C's
    // 16-byte accesses each slot four times (the least).
    static constexpr int LDS = (1 << TB) + (1 << (TB - 3));
    CK_HD static u32 slot(u32 a) { return a + 2 * (a >> 4); }
    CK_HD static u32 lds_at(int geo, u32 tid, int i) {
        const u32 a = slot((t_of(geo, tid, 0) << CL) | col_of(geo, tid, 0)) +
                      slot((t_of(geo, 0, i) << CL) | col_of(geo, 0, i));
        CK_BOUNDS(a, (u32)LDS);
        return a;
    }
    template <int GEO>
    CK_HD static void put(const u64 (&v)[8], u32 tid, u64 *lds) {
        if constexpr (GEO == 2 && EX > 0) {
#pragma unroll
            for (int i = 0; i < 8; i += 2) {
                Pair p = {v[i], v[i + 1]};
                *(Pair *)(lds + lds_at(GEO, tid, i)) = p;
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) lds[lds_at(GEO, tid, i)] = v[i];
        }
    }
    template <int GEO>
    CK_HD static void get(u64 (&v)[8], u32 tid, const u64 *lds) {
        if constexpr (GEO == 2 && EX > 0) {
#pragma unroll
            for (int i = 0; i < 8; i += 2) {
                const Pair p = *(const Pair *)(lds + lds_at(GEO, tid, i));
                v[i] = p.x;
                v[i + 1] = p.y;
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = lds[lds_at(GEO, tid, i)];
        }
    }

    // inter-pass offset of register i (geometry A): row m of column u
    CK_HD static u32 internal_off(u32 tile, u32 n1, u32 tid, int i) {
        const u32 u = (tile << CL) + col_of(0, tid, 0);
        return (bitrev(u, n1) << L) + t_of(0, tid, i);
    }
    // natural offset of register i (geometry C)
    CK_HD static u32 natural_off(u32 tile, u32 n1, u32 tid, int i) {
        return (bitrev(t_of(2, tid, i), L) << n1) + (tile << CL) + col_of(2, tid, i);
    }

    // block j of forward stage s at register i (pair bit of the stage clear)
    template <int GEO>
    CK_HD static u32 block_index(u32 tid, int i, int s) {
        return GEO == 0 ? (u32)i >> (3 - s) : t_of(GEO, tid, i) >> (L - s);
    }
    // Twiddle of register i at stage 3 GEO + k.  Geometries 0 and 1: uniform
    // over the wave, read through the scalar unit.  Geometry 2: one of the
    // thread's 2^KC - 1 entries, loaded by low_twiddles.
    struct LowTw {
        Tw t[(1 << KC) - 1];
    };
    CK_HD static LowTw low_twiddles(const Tw *tw, u32 tid) {
        LowTw l;
#pragma unroll
        for (int k = 0; k < KC; ++k)
#pragma unroll
            for (int x = 0; x < (1 << k); ++x) {
                const u32 j = block_index<2>(tid, (x << (KC - k)) << EX, 6 + k);
                CK_BOUNDS(j, 1u << (L - 1));
                l.t[(1 << k) - 1 + x] = tw[j];
            }
        return l;
    }
    template <int GEO>
    CK_HD static Tw twiddle(const Tw *tw, const LowTw &low, u32 tid, int i, int k) {
        if (GEO == 2) return low.t[(1 << k) - 1 + ((i >> EX) >> (KC - k))];
        const u32 j = block_index<GEO>(tid, i, 3 * GEO + k);
        CK_BOUNDS(j, 1u << (L - 1));
        return load_twiddle<GEO == 0 || KC + CL >= 6>(tw, j);
    }

    // Stages of one geometry; b: bounds of the residues (uniform over threads).
    template <int GEO, class Ar>
    CK_HD static void fwd(u64 (&w)[8], int (&b)[8], u32 tid, const Tw *tw, const LowTw &low, const Ar &ar) {
        constexpr int K = GEO == 2 ? KC : 3, lo = GEO == 2 ? EX : 0;
        typename Ar::V v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = Ar::from_bits(w[i]);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int bit = 1 << (lo + K - 1 - k);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (!(i & bit)) {
                    if (GEO == 0 && (i >> (3 - k)) == 0)
                        ar.ct1(v[i], v[i | bit], b[i], b[i | bit]);
                    else
                        ar.ct(v[i], v[i | bit], twiddle<GEO>(tw, low, tid, i, k), b[i], b[i | bit]);
                }
                if (!Ar::kFp && (i & 3) == 3) sched_fence();
            }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i] = Ar::to_bits(v[i]);
    }
    template <int GEO, class Ar>
    CK_HD static void inv(u64 (&w)[8], int (&b)[8], u32 tid, const Tw *tw, const LowTw &low, const Ar &ar) {
        constexpr int K = GEO == 2 ? KC : 3, lo = GEO == 2 ? EX : 0;
        typename Ar::V v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = Ar::from_bits(w[i]);
#pragma unroll
        for (int k = K - 1; k >= 0; --k) {
            const int bit = 1 << (lo + K - 1 - k);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                if (!(i & bit)) {
                    if (GEO == 0 && (i >> (3 - k)) == 0)
                        ar.gs1(v[i], v[i | bit], b[i], b[i | bit]);
                    else
                        ar.gs(v[i], v[i | bit], twiddle<GEO>(tw, low, tid, i, k), b[i], b[i | bit]);
                }
                if (!Ar::kFp && (i & 3) == 3) sched_fence();
            }
        }
        if (GEO != 0) {
#pragma unroll
            for (int i = 0; i < 8; ++i) ar.settle(v[i], b[i]);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i] = Ar::to_bits(v[i]);
    }
    // The geometry 2 stages of column group x < 2^EX alone (registers i with
    // i mod 2^EX = x are independent of the others).
    template <class Ar>
    CK_HD static void fwd_group(u64 (&w)[8], int (&b)[8], int x, const LowTw &low, const Ar &ar) {
        constexpr int M = 1 << KC;
        typename Ar::V v[M];
#pragma unroll
        for (int i = 0; i < M; ++i) v[i] = Ar::from_bits(w[(i << EX) | x]);
#pragma unroll
        for (int k = 0; k < KC; ++k) {
            const int bit = 1 << (KC - 1 - k);
#pragma unroll
            for (int i = 0; i < M; ++i)
                if (!(i & bit))
                    ar.ct(v[i], v[i | bit], low.t[(1 << k) - 1 + (i >> (KC - k))], b[(i << EX) | x],
                          b[((i | bit) << EX) | x]);
        }
#pragma unroll
        for (int i = 0; i < M; ++i) w[(i << EX) | x] = Ar::to_bits(v[i]);
    }
    // all residues at the largest bound among them (after an exchange)
    CK_HD static void level(int (&b)[8]) {
        int m = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) m = b[i] > m ? b[i] : m;
#pragma unroll
        for (int i = 0; i < 8; ++i) b[i] = m;
    }
    CK_HD static void set(int (&b)[8], int v) {
#pragma unroll
        for (int i = 0; i < 8; ++i) b[i] = v;
    }
};

}  // namespace ck
