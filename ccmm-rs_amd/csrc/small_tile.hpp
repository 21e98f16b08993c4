// Transform of a whole limb of N = 2^L <= 4096 residues in one workgroup.
//
// One launch of a few such transforms is what the smallest calls wait for: a
// workgroup has a CU to itself, so its time is the chain of loads, butterflies
// and exchanges.  Eight residues a thread (two waves on every SIMD, where
// sixteen leave one) hide the latencies in each other; every twiddle of the
// later rounds is requested before the first butterfly; one barrier per
// exchange (two LDS buffers).
//
// Rounds A, B, C, D of stages 0-2, 3-5, 6-8 and the L - 9 left; register i
// holds bits PR .. PR + 2 of the position t, the thread number the others in
// order.  Natural order (n = bitrev(t)) is one more exchange: E.
#pragma once
#include "row_tile.hpp"

namespace ck {

template <int L>
struct SmallTile {
    static_assert(L >= 10 && L <= 12, "single-pass degrees");
    static constexpr u32 THREADS = 1u << (L - 3);
    static constexpr int LDS = (1 << L) + (1 << (L - 6));

    CK_HD static constexpr int pos(int r) { return r < 3 ? L - 3 - 3 * r : 0; }
    CK_HD static constexpr int stages(int r) { return r < 3 ? 3 : L - 9; }
    CK_HD static u32 t_of(int r, u32 tid, int i) {
        const int p = pos(r);
        return (tid & ((1u << p) - 1)) | ((u32)i << p) | ((tid >> p) << (p + 3));
    }
    // one residue of padding per 64: conflict-free or two-way in every round
    CK_HD static u32 slot(u32 t) {
        const u32 s = t + (t >> 6);
        CK_BOUNDS(s, (u32)LDS);
        return s;
    }
    template <int R>
    CK_HD static void put(const u64 (&v)[8], u32 tid, u64 *lds) {
#pragma unroll
        for (int i = 0; i < 8; ++i) lds[slot(t_of(R, tid, i))] = v[i];
    }
    template <int R>
    CK_HD static void get(u64 (&v)[8], u32 tid, const u64 *lds) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = lds[slot(t_of(R, tid, i))];
    }
    // natural position of register i: tid + i THREADS
    CK_HD static void put_natural(const u64 (&v)[8], u32 tid, u64 *lds) {
#pragma unroll
        for (int i = 0; i < 8; ++i) lds[slot(bitrev(tid + i * THREADS, L))] = v[i];
    }
    CK_HD static void get_natural(u64 (&v)[8], u32 tid, const u64 *lds) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = lds[slot(bitrev(tid + i * THREADS, L))];
    }

    // The thread's twiddles of round R, K stages on the lower K register bits:
    // stage k (bit K - 1 - k) has one per value of the register bits above it.
    struct Tws {
        Tw t[7];
    };
    template <int R>
    CK_HD static constexpr int entry(int i, int k) {
        return (((1 << k) - 1) << (3 - stages(R))) + (i >> (stages(R) - k));
    }
    template <int R>
    CK_HD static Tws twiddles(const Tw *tw, u32 tid) {
        constexpr int K = stages(R);
        Tws w{};
#pragma unroll
        for (int k = 0; k < K; ++k)
#pragma unroll
            for (int i = 0; i < 8; i += 1 << (K - k)) {
                const u32 j = (1u << (3 * R + k)) + (t_of(R, tid, i) >> (L - 3 * R - k));
                CK_BOUNDS(j, 1u << L);
                // uniform over a wave in round A, and in B where 64 threads
                // share the bits above the round's
                w.t[entry<R>(i, k)] = R == 0 || (R == 1 && pos(1) >= 6) ? load_twiddle<true>(tw, j) : tw[j];
            }
        return w;
    }
    template <int R>
    CK_HD static constexpr int bit_of(int k) {
        return 1 << (stages(R) - 1 - k);
    }
    template <int R, class Ar>
    CK_HD static void fwd(u64 (&w)[8], int (&b)[8], const Tws &tw, const Ar &ar) {
        typename Ar::V v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = Ar::from_bits(w[i]);
#pragma unroll
        for (int k = 0; k < stages(R); ++k) {
            const int bit = bit_of<R>(k);
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (!(i & bit)) ar.ct(v[i], v[i | bit], tw.t[entry<R>(i, k)], b[i], b[i | bit]);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i] = Ar::to_bits(v[i]);
    }
    template <int R, class Ar>
    CK_HD static void inv(u64 (&w)[8], int (&b)[8], const Tws &tw, const Ar &ar) {
        typename Ar::V v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = Ar::from_bits(w[i]);
#pragma unroll
        for (int k = stages(R) - 1; k >= 0; --k) {
            const int bit = bit_of<R>(k);
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (!(i & bit)) ar.gs(v[i], v[i | bit], tw.t[entry<R>(i, k)], b[i], b[i | bit]);
        }
        if (R != 0) {
#pragma unroll
            for (int i = 0; i < 8; ++i) ar.settle(v[i], b[i]);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i] = Ar::to_bits(v[i]);
    }
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
