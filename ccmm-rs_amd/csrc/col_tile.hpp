// Column-pass tile of the fused kernels: stages 0 .. n1-1 of a two-pass
// transform (the merged negacyclic network of ntt_tile.hpp) over 2^(12-K1)
// columns of 2^K1 residues, with the bound-tracked arithmetic of row_tile.hpp.
// B = 4: 16 residues per thread in 256 threads, two rounds and one LDS exchange:
//   geometry 0: the top four bits of t in registers (twiddles are constants of
//               the unrolled code, read through the scalar unit);
//   geometry 1: the low K1 - 4 bits of t and the top 8 - K1 column bits.
// Lanes walk at least 16 consecutive columns in both, so every access to HBM
// is whole 128-byte runs and the natural order is kept: a tile reads and
// writes the same positions.
// B = 3: 8 residues in 512 threads, two rounds (K1 = 6) or three, the last with
// the low bits of t and the top column bits again: twice the waves for launches
// of few tiles, where a wave's own latency is what counts.
#pragma once
#include "row_tile.hpp"

namespace ck {

template <int K1, int B = 4>
struct ColTile {
    static constexpr int K = K1, M = 1 << B, CL = 12 - K1, ROUNDS = (K1 + B - 1) / B;
    static constexpr u32 THREADS = 4096u >> B;
    static_assert(K1 >= 6 && K1 <= 8 && ROUNDS <= 3, "columns of 64 .. 256 residues");
    static constexpr int LAST = ROUNDS - 1, KB = K1 - B * LAST;  // last geometry, its stages
    static constexpr int CB = CL - (B - KB);                     // its column bits in the thread number

    CK_HD static constexpr int stages(int geo) { return geo == LAST ? KB : B; }
    CK_HD static u32 t_of(int geo, u32 tid, int i) {
        if (geo == LAST) return ((tid >> CB) << KB) | ((u32)i & ((1u << KB) - 1));
        const int p = K1 - B * (geo + 1);
        const u32 r = tid >> CL;
        return (r & ((1u << p) - 1)) | ((u32)i << p) | ((r >> p) << (p + B));
    }
    CK_HD static u32 col_of(int geo, u32 tid, int i) {
        if (geo == LAST) return (tid & ((1u << CB) - 1)) | (((u32)i >> KB) << CB);
        return tid & ((1u << CL) - 1);
    }
    CK_HD static u32 lds_at(int geo, u32 tid, int i) {
        const u32 a = row_swizzle((t_of(geo, tid, 0) << CL) | col_of(geo, tid, 0)) ^
                      row_swizzle((t_of(geo, 0, i) << CL) | col_of(geo, 0, i));
        CK_BOUNDS(a, 4096u);
        return a;
    }
    template <int GEO>
    CK_HD static void put(const u64 (&v)[M], u32 tid, u64 *lds) {
#pragma unroll
        for (int i = 0; i < M; ++i) lds[lds_at(GEO, tid, i)] = v[i];
    }
    template <int GEO>
    CK_HD static void get(u64 (&v)[M], u32 tid, const u64 *lds) {
#pragma unroll
        for (int i = 0; i < M; ++i) v[i] = lds[lds_at(GEO, tid, i)];
    }
    // position of register i in the limb (n2 = log2 of the row length)
    template <int GEO>
    CK_HD static u32 offset(u32 tile, u32 n2, u32 tid, int i) {
        return (t_of(GEO, tid, i) << n2) + (tile << CL) + col_of(GEO, tid, i);
    }

    // offset(.., i) - offset(.., 0): the same in every thread
    template <int GEO>
    CK_HD static u32 step(u32 n2, int i) {
        return (t_of(GEO, 0, i) << n2) + col_of(GEO, 0, i);
    }
    template <int GEO>
    CK_HD static Tw twiddle(const Tw *tw, u32 tid, int i, int s) {
        const u32 j = GEO == 0 ? (u32)i >> (B - s) : t_of(GEO, tid, i) >> (K1 - s);
        const u32 k = (1u << s) + j;
        CK_BOUNDS(k, 1u << K1);
        return GEO == 0 ? load_twiddle<true>(tw, k) : load_twiddle<false>(tw, k);
    }
    template <int GEO, class Ar>
    CK_HD static void fwd(u64 (&w)[M], int (&b)[M], u32 tid, const Tw *tw, const Ar &ar) {
        constexpr int K = stages(GEO), s0 = GEO * B;
        typename Ar::V v[M];
#pragma unroll
        for (int i = 0; i < M; ++i) v[i] = Ar::from_bits(w[i]);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int bit = 1 << (K - 1 - k);
#pragma unroll
            for (int i = 0; i < M; ++i) {
                if (!(i & bit)) ar.ct(v[i], v[i | bit], twiddle<GEO>(tw, tid, i, s0 + k), b[i], b[i | bit]);
                if (!Ar::kFp && (i & 3) == 3) sched_fence();
            }
        }
#pragma unroll
        for (int i = 0; i < M; ++i) w[i] = Ar::to_bits(v[i]);
    }
    template <int GEO, class Ar>
    CK_HD static void inv(u64 (&w)[M], int (&b)[M], u32 tid, const Tw *tw, const Ar &ar) {
        constexpr int K = stages(GEO), s0 = GEO * B;
        typename Ar::V v[M];
#pragma unroll
        for (int i = 0; i < M; ++i) v[i] = Ar::from_bits(w[i]);
#pragma unroll
        for (int k = K - 1; k >= 0; --k) {
            const int bit = 1 << (K - 1 - k);
#pragma unroll
            for (int i = 0; i < M; ++i) {
                if (!(i & bit)) ar.gs(v[i], v[i | bit], twiddle<GEO>(tw, tid, i, s0 + k), b[i], b[i | bit]);
                if (!Ar::kFp && (i & 3) == 3) sched_fence();
            }
        }
        if (GEO != 0) {
#pragma unroll
            for (int i = 0; i < M; ++i) ar.settle(v[i], b[i]);
        }
#pragma unroll
        for (int i = 0; i < M; ++i) w[i] = Ar::to_bits(v[i]);
    }
    CK_HD static void level(int (&b)[M]) {
        int m = 0;
#pragma unroll
        for (int i = 0; i < M; ++i) m = b[i] > m ? b[i] : m;
#pragma unroll
        for (int i = 0; i < M; ++i) b[i] = m;
    }
    CK_HD static void set(int (&b)[M], int v) {
#pragma unroll
        for (int i = 0; i < M; ++i) b[i] = v;
    }
};

}  // namespace ck
