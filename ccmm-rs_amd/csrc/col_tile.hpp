// Column-pass tile of the fused kernels: stages 0 .. n1-1 of a two-pass
// transform (the merged negacyclic network of ntt_tile.hpp) over 2^(12-K1)
// columns of 2^K1 residues, with the bound-tracked arithmetic of row_tile.hpp.
// 16 residues per thread in 256 threads, two rounds and one LDS exchange:
//   geometry 0: the top four bits of t in registers (twiddles are constants of
//               the unrolled code, read through the scalar unit);
//   geometry 1: the low K1 - 4 bits of t and the top 8 - K1 column bits.
// Lanes walk at least 16 consecutive columns in both, so every access to HBM
// is whole 128-byte runs and the natural order is kept: a tile reads and
// writes the same positions.
#pragma once
#include "row_tile.hpp"

namespace ck {

template <int K1>
struct ColTile {
    static constexpr int CL = 12 - K1, KB = K1 - 4;
    static_assert(K1 >= 6 && K1 <= 8, "columns of 64 .. 256 residues");

    CK_HD static u32 t_of(int geo, u32 tid, int i) {
        if (geo == 0) return (tid >> CL) | ((u32)i << KB);
        return ((tid >> 4) << KB) | ((u32)i & ((1u << KB) - 1));
    }
    CK_HD static u32 col_of(int geo, u32 tid, int i) {
        if (geo == 0) return tid & ((1u << CL) - 1);
        return (tid & 15u) | (((u32)i >> KB) << 4);
    }
    CK_HD static u32 lds_at(int geo, u32 tid, int i) {
        const u32 a = row_swizzle((t_of(geo, tid, 0) << CL) | col_of(geo, tid, 0)) ^
                      row_swizzle((t_of(geo, 0, i) << CL) | col_of(geo, 0, i));
        CK_BOUNDS(a, 4096u);
        return a;
    }
    template <int GEO>
    CK_HD static void put(const u64 (&v)[16], u32 tid, u64 *lds) {
#pragma unroll
        for (int i = 0; i < 16; ++i) lds[lds_at(GEO, tid, i)] = v[i];
    }
    template <int GEO>
    CK_HD static void get(u64 (&v)[16], u32 tid, const u64 *lds) {
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = lds[lds_at(GEO, tid, i)];
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
        const u32 j = GEO == 0 ? (u32)i >> (4 - s) : t_of(1, tid, i) >> (K1 - s);
        const u32 k = (1u << s) + j;
        CK_BOUNDS(k, 1u << K1);
        return GEO == 0 ? load_twiddle<true>(tw, k) : load_twiddle<false>(tw, k);
    }
    template <int GEO, class Ar>
    CK_HD static void fwd(u64 (&w)[16], int (&b)[16], u32 tid, const Tw *tw, const Ar &ar) {
        constexpr int K = GEO == 0 ? 4 : KB, s0 = GEO * 4;
        typename Ar::V v[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = Ar::from_bits(w[i]);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int bit = 1 << (K - 1 - k);
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                if (!(i & bit)) ar.ct(v[i], v[i | bit], twiddle<GEO>(tw, tid, i, s0 + k), b[i], b[i | bit]);
                if (!Ar::kFp && (i & 3) == 3) sched_fence();
            }
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) w[i] = Ar::to_bits(v[i]);
    }
    template <int GEO, class Ar>
    CK_HD static void inv(u64 (&w)[16], int (&b)[16], u32 tid, const Tw *tw, const Ar &ar) {
        constexpr int K = GEO == 0 ? 4 : KB, s0 = GEO * 4;
        typename Ar::V v[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) v[i] = Ar::from_bits(w[i]);
#pragma unroll
        for (int k = K - 1; k >= 0; --k) {
            const int bit = 1 << (K - 1 - k);
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                if (!(i & bit)) ar.gs(v[i], v[i | bit], twiddle<GEO>(tw, tid, i, s0 + k), b[i], b[i | bit]);
                if (!Ar::kFp && (i & 3) == 3) sched_fence();
            }
        }
        if (GEO != 0) {
#pragma unroll
            for (int i = 0; i < 16; ++i) ar.settle(v[i], b[i]);
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) w[i] = Ar::to_bits(v[i]);
    }
    CK_HD static void level(int (&b)[16]) {
        int m = 0;
#pragma unroll
        for (int i = 0; i < 16; ++i) m = b[i] > m ? b[i] : m;
#pragma unroll
        for (int i = 0; i < 16; ++i) b[i] = m;
    }
    CK_HD static void set(int (&b)[16], int v) {
#pragma unroll
        for (int i = 0; i < 16; ++i) b[i] = v;
    }
};

}  // namespace ck
