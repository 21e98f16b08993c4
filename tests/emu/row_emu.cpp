// CPU build of the fused row tiles (row_tile.hpp, the source of the gfx950
// kernels), every LDS, HBM and twiddle index bounds-checked.  Test
// infrastructure only.
#define CK_CHECK_BOUNDS 1
#include <cstring>
#include <vector>

#include "../../ccmm-rs_amd/csrc/host_math.hpp"
#include "../../ccmm-rs_amd/csrc/ntt_pass.hpp"
#include "../../ccmm-rs_amd/csrc/col_tile.hpp"
#include "../../ccmm-rs_amd/csrc/row_sums.hpp"
#include "../../ccmm-rs_amd/csrc/small_tile.hpp"

using namespace ck;

namespace {

struct Limb {
    u64 q;
    u32 logn;
    bool fp;
    std::vector<uint64_t> fwd, inv;
    Limb(u64 q_, u32 logn_) : q(q_), logn(logn_), fp(q_ < host::kFpModulusBound) {
        const u64 psi = host::negacyclic_root(q, 1ull << logn);
        if (fp) {
            host::twiddle_table_fp(q, psi, logn, fwd);
            host::twiddle_table_fp(q, host::invmod(psi, q), logn, inv);
        } else {
            host::twiddle_table(q, psi, logn, fwd);
            host::twiddle_table(q, host::invmod(psi, q), logn, inv);
        }
    }
    const Tw *tw(bool forward) const { return reinterpret_cast<const Tw *>((forward ? fwd : inv).data()); }
    // psi^((2u+1) t) (or its inverse), as build_row_products gathers it
    Tw row_product(u32 off, bool forward) const {
        const u32 n2 = ntt_n2(logn), n1 = logn - n2, N = 1u << logn;
        const u32 u = bitrev(off >> n2, n1), t = off & ((1u << n2) - 1);
        const u32 e = ((2 * u + 1) * t) & (2 * N - 1);
        const Tw w = tw(forward)[bitrev(e & (N - 1), logn)];
        if (e < N) return w;
        if (fp) return Tw{f64_as_u64((double)q - u64_as_f64(w.w)), 0};
        return Tw{q - w.w, ~w.wq};
    }
};

RowFp::Z z_of(const Tw &w, const RowFp &) { return u64_as_f64(w.w); }
RowInt::Z z_of(const Tw &w, const RowInt &) { return w; }

u64 canonical(u64 x, const RowFp &ar) { return fp_canonical(u64_as_f64(x), ar.q, ar.qinv); }
u64 canonical(u64 x, const RowInt &ar) { return x % ar.q; }
u64 lazy(u64 x, const RowFp &) { return f64_as_u64((double)x); }
u64 lazy(u64 x, const RowInt &) { return x; }

// forward: inter-pass data -> natural-order values; inverse the other way.
template <int L, int TB, class Ar>
void row_pass(const Limb &p, const Ar &ar, const u64 *in, u64 *out, bool forward) {
    typedef RowTile<L, TB> R;
    const u32 n1 = p.logn - L;
    static u64 v[R::THREADS][8];
    alignas(16) static u64 lds[R::LDS];
    for (u32 tile = 0; tile < (1u << (p.logn - TB)); ++tile) {
        int b[8], bx[8];
        auto each = [&](auto &&f) {
            for (u32 tid = 0; tid < R::THREADS; ++tid) f(tid);
        };
        auto rounds = [&](auto &&f) {
            for (u32 tid = 0; tid < R::THREADS; ++tid) {
                std::memcpy(bx, b, sizeof b);
                f(tid);
            }
            std::memcpy(b, bx, sizeof b);
        };
        const Tw *tw = p.tw(forward);
        const typename R::LowTw none{};
        std::memset(lds, 0xA5, sizeof lds);
        if (forward) {
            each([&](u32 t) {
                for (int i = 0; i < 8; ++i) {
                    const u32 o = R::internal_off(tile, n1, t, i);
                    CK_BOUNDS(o, 1u << p.logn);
                    v[t][i] = ar.times(lazy(in[o], ar), z_of(p.row_product(o, true), ar));
                }
            });
            R::set(b, Ar::kZ);
            rounds([&](u32 t) { R::template fwd<0>(v[t], bx, t, tw, none, ar); });
            each([&](u32 t) { R::template put<0>(v[t], t, lds); });
            each([&](u32 t) { R::template get<1>(v[t], t, lds); });
            R::level(b);
            rounds([&](u32 t) { R::template fwd<1>(v[t], bx, t, tw, none, ar); });
            each([&](u32 t) { R::template put<1>(v[t], t, lds); });
            each([&](u32 t) { R::template get<2>(v[t], t, lds); });
            R::level(b);
            rounds([&](u32 t) {
                for (int x = 0; x < (1 << R::EX); ++x) R::fwd_group(v[t], bx, x, R::low_twiddles(tw, t), ar);
            });
            each([&](u32 t) {
                for (int i = 0; i < 8; ++i) {
                    const u32 o = R::natural_off(tile, n1, t, i);
                    CK_BOUNDS(o, 1u << p.logn);
                    out[o] = canonical(v[t][i], ar);
                }
            });
        } else {
            each([&](u32 t) {
                for (int i = 0; i < 8; ++i) {
                    const u32 o = R::natural_off(tile, n1, t, i);
                    CK_BOUNDS(o, 1u << p.logn);
                    // a centered double in half a q, as the kernels reduce their sums
                    v[t][i] = Ar::kFp ? f64_as_u64((double)in[o] - (in[o] > p.q / 2 ? (double)p.q : 0.0)) : in[o];
                }
            });
            R::set(b, 1);
            rounds([&](u32 t) { R::template inv<2>(v[t], bx, t, tw, R::low_twiddles(tw, t), ar); });
            each([&](u32 t) { R::template put<2>(v[t], t, lds); });
            each([&](u32 t) { R::template get<1>(v[t], t, lds); });
            R::level(b);
            rounds([&](u32 t) { R::template inv<1>(v[t], bx, t, tw, none, ar); });
            each([&](u32 t) { R::template put<1>(v[t], t, lds); });
            each([&](u32 t) { R::template get<0>(v[t], t, lds); });
            R::level(b);
            rounds([&](u32 t) { R::template inv<0>(v[t], bx, t, tw, none, ar); });
            each([&](u32 t) {
                for (int i = 0; i < 8; ++i) {
                    const u32 o = R::internal_off(tile, n1, t, i);
                    CK_BOUNDS(o, 1u << p.logn);
                    out[o] = canonical(ar.times(v[t][i], z_of(p.row_product(o, false), ar)), ar);
                }
            });
        }
    }
}

// forward: coefficients -> inter-pass residues (canonical here), without the
// row products; inverse the other way, times N^-1.
template <int K1, int B, class Ar>
void col_pass(const Limb &p, const Ar &ar, const u64 *in, u64 *out, bool forward, int bound) {
    typedef ColTile<K1, B> C;
    const u32 n2 = p.logn - K1;
    const u64 q = p.q, ninv = host::invmod((1ull << p.logn) % q, q), ninv_q = host::shoup_quotient(ninv, q);
    static u64 v[C::THREADS][C::M];
    static u64 lds[4096];
    for (u32 tile = 0; tile < (1u << (p.logn - 12)); ++tile) {
        int b[C::M], bx[C::M];
        auto each = [&](auto &&f) {
            for (u32 tid = 0; tid < C::THREADS; ++tid) f(tid);
        };
        auto rounds = [&](auto &&f) {
            for (u32 tid = 0; tid < C::THREADS; ++tid) {
                std::memcpy(bx, b, sizeof b);
                f(tid);
            }
            std::memcpy(b, bx, sizeof b);
        };
        const Tw *tw = p.tw(forward);
        std::memset(lds, 0xA5, sizeof lds);
        C::set(b, bound);
        if (forward) {
            each([&](u32 t) {
                for (int i = 0; i < C::M; ++i) {
                    const u32 o = C::template offset<0>(tile, n2, t, i);
                    CK_BOUNDS(o, 1u << p.logn);
                    v[t][i] = lazy(in[o], ar);
                }
            });
            rounds([&](u32 t) { C::template fwd<0>(v[t], bx, t, tw, ar); });
            each([&](u32 t) { C::template put<0>(v[t], t, lds); });
            each([&](u32 t) { C::template get<1>(v[t], t, lds); });
            C::level(b);
            rounds([&](u32 t) { C::template fwd<1>(v[t], bx, t, tw, ar); });
            if constexpr (C::LAST == 2) {
                each([&](u32 t) { C::template put<1>(v[t], t, lds); });
                each([&](u32 t) { C::template get<2>(v[t], t, lds); });
                C::level(b);
                rounds([&](u32 t) { C::template fwd<2>(v[t], bx, t, tw, ar); });
            }
            each([&](u32 t) {
                for (int i = 0; i < C::M; ++i) {
                    const u32 o = C::template offset<C::LAST>(tile, n2, t, i);
                    CK_BOUNDS(o, 1u << p.logn);
                    out[o] = canonical(v[t][i], ar);
                }
            });
        } else {
            each([&](u32 t) {
                for (int i = 0; i < C::M; ++i) v[t][i] = lazy(in[C::template offset<C::LAST>(tile, n2, t, i)], ar);
            });
            if constexpr (C::LAST == 2) {
                rounds([&](u32 t) { C::template inv<2>(v[t], bx, t, tw, ar); });
                each([&](u32 t) { C::template put<2>(v[t], t, lds); });
                each([&](u32 t) { C::template get<1>(v[t], t, lds); });
                C::level(b);
            }
            rounds([&](u32 t) { C::template inv<1>(v[t], bx, t, tw, ar); });
            each([&](u32 t) { C::template put<1>(v[t], t, lds); });
            each([&](u32 t) { C::template get<0>(v[t], t, lds); });
            C::level(b);
            rounds([&](u32 t) { C::template inv<0>(v[t], bx, t, tw, ar); });
            each([&](u32 t) {
                for (int i = 0; i < C::M; ++i) {
                    const u32 o = C::template offset<0>(tile, n2, t, i);
                    CK_BOUNDS(o, 1u << p.logn);
                    out[o] = shoup(canonical(v[t][i], ar), ninv, ninv_q, q);
                }
            });
        }
    }
}

// TB: 12, or 11 for the halved tiles of small launches
template <int TB = 12, class Ar>
int run(const Limb &p, const Ar &ar, const u64 *in, u64 *out, bool forward) {
    switch (ntt_n2(p.logn)) {
        case 7: row_pass<7, TB>(p, ar, in, out, forward); return 0;
        case 8: row_pass<8, TB>(p, ar, in, out, forward); return 0;
        case 9: row_pass<9, TB>(p, ar, in, out, forward); return 0;
        default: return -1;
    }
}

// A whole transform of a single-pass degree, natural order both ways.
template <int L, class Ar>
void small_pass(const Limb &p, const Ar &ar, const u64 *in, u64 *out, bool forward, int bound) {
    typedef SmallTile<L> S;
    const u64 q = p.q, ninv = host::invmod((1ull << L) % q, q), ninv_q = host::shoup_quotient(ninv, q);
    static u64 v[S::THREADS][8];
    static u64 lds[2][S::LDS];
    int b[8], bx[8];
    auto each = [&](auto &&f) {
        for (u32 tid = 0; tid < S::THREADS; ++tid) f(tid);
    };
    auto rounds = [&](auto &&f) {
        for (u32 tid = 0; tid < S::THREADS; ++tid) {
            std::memcpy(bx, b, sizeof b);
            f(tid);
        }
        std::memcpy(b, bx, sizeof b);
    };
    const Tw *tw = p.tw(forward);
    std::memset(lds, 0xA5, sizeof lds);
    each([&](u32 t) {
        for (int i = 0; i < 8; ++i) v[t][i] = lazy(in[t + i * S::THREADS], ar);
    });
    S::set(b, bound);
    // the kernels' exchanges: the buffers take turns
    if (forward) {
        rounds([&](u32 t) { S::template fwd<0>(v[t], bx, S::template twiddles<0>(tw, t), ar); });
        each([&](u32 t) { S::template put<0>(v[t], t, lds[0]); });
        each([&](u32 t) { S::template get<1>(v[t], t, lds[0]); });
        S::level(b);
        rounds([&](u32 t) { S::template fwd<1>(v[t], bx, S::template twiddles<1>(tw, t), ar); });
        each([&](u32 t) { S::template put<1>(v[t], t, lds[1]); });
        each([&](u32 t) { S::template get<2>(v[t], t, lds[1]); });
        S::level(b);
        rounds([&](u32 t) { S::template fwd<2>(v[t], bx, S::template twiddles<2>(tw, t), ar); });
        each([&](u32 t) { S::template put<2>(v[t], t, lds[0]); });
        each([&](u32 t) { S::template get<3>(v[t], t, lds[0]); });
        S::level(b);
        rounds([&](u32 t) { S::template fwd<3>(v[t], bx, S::template twiddles<3>(tw, t), ar); });
        each([&](u32 t) {
            for (int i = 0; i < 8; ++i) v[t][i] = canonical(v[t][i], ar);
            S::template put<3>(v[t], t, lds[1]);
        });
        each([&](u32 t) { S::get_natural(v[t], t, lds[1]); });
    } else {
        each([&](u32 t) { S::put_natural(v[t], t, lds[0]); });
        each([&](u32 t) { S::template get<3>(v[t], t, lds[0]); });
        rounds([&](u32 t) { S::template inv<3>(v[t], bx, S::template twiddles<3>(tw, t), ar); });
        each([&](u32 t) { S::template put<3>(v[t], t, lds[1]); });
        each([&](u32 t) { S::template get<2>(v[t], t, lds[1]); });
        S::level(b);
        rounds([&](u32 t) { S::template inv<2>(v[t], bx, S::template twiddles<2>(tw, t), ar); });
        each([&](u32 t) { S::template put<2>(v[t], t, lds[0]); });
        each([&](u32 t) { S::template get<1>(v[t], t, lds[0]); });
        S::level(b);
        rounds([&](u32 t) { S::template inv<1>(v[t], bx, S::template twiddles<1>(tw, t), ar); });
        each([&](u32 t) { S::template put<1>(v[t], t, lds[1]); });
        each([&](u32 t) { S::template get<0>(v[t], t, lds[1]); });
        S::level(b);
        rounds([&](u32 t) { S::template inv<0>(v[t], bx, S::template twiddles<0>(tw, t), ar); });
        each([&](u32 t) {
            for (int i = 0; i < 8; ++i) v[t][i] = shoup(canonical(v[t][i], ar), ninv, ninv_q, q);
        });
    }
    each([&](u32 t) {
        for (int i = 0; i < 8; ++i) out[t + i * S::THREADS] = v[t][i];
    });
}

}  // namespace

// The row pass alone over one limb: forward takes canonical inter-pass
// residues (row m = bitrev(u) at m N2) to natural-order values, inverse the
// values back (times nothing: the column pass scales by N^-1).
extern "C" int emu_row_pass(const uint64_t *in, uint64_t *out, uint64_t q, uint32_t logn, int forward) {
    if (logn < 13 || logn > 17 || q >= kLazyModulusBound) return -1;
    if (!host::negacyclic_root(q, 1ull << logn)) return -2;
    const Limb p(q, logn);
    if (p.fp) return run(p, RowFp{(double)q, 1.0 / (double)q}, in, out, forward != 0);
    return run(p, RowInt{q}, in, out, forward != 0);
}

// Column passes: the kernels' input bounds (kColFpIn, kColIntIn, row products)
template <int B = 4, class Ar>
static int col_run(const Limb &p, const Ar &ar, const u64 *in, u64 *out, bool forward) {
    // canonical residues enter an inverse as 2 units of 0.52 q (FP64)
    const int bound = forward ? (Ar::kFp ? 16 : 4) : (Ar::kFp ? 2 : 3);
    switch (ntt_n1(p.logn)) {
        case 6: col_pass<6, B>(p, ar, in, out, forward, bound); return 0;
        case 7: col_pass<7, B>(p, ar, in, out, forward, bound); return 0;
        case 8: col_pass<8, B>(p, ar, in, out, forward, bound); return 0;
        default: return -1;
    }
}

template <int TB, int B>
static int fused_ntt(const uint64_t *in, uint64_t *out, uint64_t q, uint32_t logn, int forward) {
    if (logn < 13 || logn > 17 || q >= kLazyModulusBound) return -1;
    if (!host::negacyclic_root(q, 1ull << logn)) return -2;
    const Limb p(q, logn);
    std::vector<uint64_t> mid(1ull << logn);
    auto go = [&](const auto &ar) {
        int rc = forward ? col_run<B>(p, ar, in, mid.data(), true) : run<TB>(p, ar, in, mid.data(), false);
        if (rc) return rc;
        return forward ? run<TB>(p, ar, mid.data(), out, true) : col_run<B>(p, ar, mid.data(), out, false);
    };
    return p.fp ? go(RowFp{(double)q, 1.0 / (double)q}) : go(RowInt{q});
}

// A whole transform by column and row tiles: forward canonical coefficients to
// natural-order values, inverse back.
extern "C" int emu_fused_ntt(const uint64_t *in, uint64_t *out, uint64_t q, uint32_t logn, int forward) {
    return fused_ntt<12, 4>(in, out, q, logn, forward);
}
// The same by the tiles of small launches.
extern "C" int emu_fused_ntt_halved(const uint64_t *in, uint64_t *out, uint64_t q, uint32_t logn, int forward) {
    return fused_ntt<11, 3>(in, out, q, logn, forward);
}

// A transform of a single-pass degree at the kernels' largest input bounds.
extern "C" int emu_small_ntt(const uint64_t *in, uint64_t *out, uint64_t q, uint32_t logn, int forward) {
    if (logn < 10 || logn > 12 || q >= kLazyModulusBound) return -1;
    if (!host::negacyclic_root(q, 1ull << logn)) return -2;
    const Limb p(q, logn);
    auto go = [&](const auto &ar, int bound) {
        switch (logn) {
            case 10: small_pass<10>(p, ar, in, out, forward, bound); break;
            case 11: small_pass<11>(p, ar, in, out, forward, bound); break;
            default: small_pass<12>(p, ar, in, out, forward, bound); break;
        }
        return 0;
    };
    return p.fp ? go(RowFp{(double)q, 1.0 / (double)q}, forward ? 16 : 2) : go(RowInt{q}, forward ? 4 : 3);
}

// sum_t c_t w_t mod q of a gadget block as the column pass and ModUp form it:
// the FP64 remainder as an integer, or the integer one shifted by q.
extern "C" int64_t emu_block_sum(int fp, const uint64_t *c, const uint64_t *w, int n, uint64_t q) {
    auto go = [&](auto s) {
        for (int t = 0; t < n; ++t) s.add(c[t] | kDigitBias, w[t], (double)w[t] / (double)q);
        return s.value(q);
    };
    if (!fp) return (int64_t)go(BlockSum<false>{});
    return (int64_t)u64_as_f64(go(BlockSum<true>{}));
}

// sum_j y_j w_j of a key product as the row kernels form it; *peak: the
// largest sum met (FP64: its magnitude), before any reduction.
extern "C" int64_t emu_key_sum(int fp, const int64_t *y, const uint64_t *w, int n, uint64_t q, uint64_t *peak) {
    *peak = 0;
    if (fp) {
        const SumFp sum{(double)q, 1.0 / (double)q};
        double s = 0;
        for (int j = 0; j < n; ++j) {
            sum.mac(s, f64_as_u64((double)y[j]), w[j]);
            const uint64_t m = (uint64_t)__builtin_fabs(s);
            *peak = m > *peak ? m : *peak;
            if (SumFp::full(j) && j + 1 < n) s = sum.reduced(s);
        }
        return (int64_t)u64_as_f64(sum.total(s));
    }
    uint64_t br_hi, br_lo;
    host::barrett(q, br_hi, br_lo);
    const SumInt sum(q, br_hi, br_lo);
    uint64_t s = 0;
    for (int j = 0; j < n; ++j) {
        sum.mac(s, (uint64_t)y[j], w[j]);
        *peak = s > *peak ? s : *peak;
        if (SumInt::full(j) && j + 1 < n) s = sum.reduced(s);
    }
    return (int64_t)sum.total(s);
}

// shoup_lazy3 at y w mod q: the residue it returns (before any reduction)
extern "C" uint64_t emu_shoup_lazy3(uint64_t y, uint64_t w, uint64_t q) {
    return shoup_lazy3(y, w, host::shoup_quotient(w, q), q);
}
