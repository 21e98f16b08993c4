// CPU build of the fused row tiles (row_tile.hpp, the source of the gfx950
// kernels), every LDS, HBM and twiddle index bounds-checked.  Test
// infrastructure only.
#define CK_CHECK_BOUNDS 1
#include <cstring>
#include <vector>

#include "../../ccmm-rs_amd/csrc/host_math.hpp"
#include "../../ccmm-rs_amd/csrc/ntt_pass.hpp"
#include "../../ccmm-rs_amd/csrc/col_tile.hpp"

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
template <int L, class Ar>
void row_pass(const Limb &p, const Ar &ar, const u64 *in, u64 *out, bool forward) {
    typedef RowTile<L> R;
    const u32 n1 = p.logn - L;
    static u64 v[512][8];
    alignas(16) static u64 lds[RowTile<L>::LDS];
    for (u32 tile = 0; tile < (1u << (p.logn - 12)); ++tile) {
        int b[8], bx[8];
        auto each = [&](auto &&f) {
            for (u32 tid = 0; tid < 512; ++tid) f(tid);
        };
        auto rounds = [&](auto &&f) {
            for (u32 tid = 0; tid < 512; ++tid) {
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
template <int K1, class Ar>
void col_pass(const Limb &p, const Ar &ar, const u64 *in, u64 *out, bool forward, int bound) {
    typedef ColTile<K1> C;
    const u32 n2 = p.logn - K1;
    const u64 q = p.q, ninv = host::invmod((1ull << p.logn) % q, q), ninv_q = host::shoup_quotient(ninv, q);
    static u64 v[256][16];
    static u64 lds[4096];
    for (u32 tile = 0; tile < (1u << (p.logn - 12)); ++tile) {
        int b[16], bx[16];
        auto each = [&](auto &&f) {
            for (u32 tid = 0; tid < 256; ++tid) f(tid);
        };
        auto rounds = [&](auto &&f) {
            for (u32 tid = 0; tid < 256; ++tid) {
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
                for (int i = 0; i < 16; ++i) {
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
            each([&](u32 t) {
                for (int i = 0; i < 16; ++i) {
                    const u32 o = C::template offset<1>(tile, n2, t, i);
                    CK_BOUNDS(o, 1u << p.logn);
                    out[o] = canonical(v[t][i], ar);
                }
            });
        } else {
            each([&](u32 t) {
                for (int i = 0; i < 16; ++i) v[t][i] = lazy(in[C::template offset<1>(tile, n2, t, i)], ar);
            });
            rounds([&](u32 t) { C::template inv<1>(v[t], bx, t, tw, ar); });
            each([&](u32 t) { C::template put<1>(v[t], t, lds); });
            each([&](u32 t) { C::template get<0>(v[t], t, lds); });
            C::level(b);
            rounds([&](u32 t) { C::template inv<0>(v[t], bx, t, tw, ar); });
            each([&](u32 t) {
                for (int i = 0; i < 16; ++i) {
                    const u32 o = C::template offset<0>(tile, n2, t, i);
                    CK_BOUNDS(o, 1u << p.logn);
                    out[o] = shoup(canonical(v[t][i], ar), ninv, ninv_q, q);
                }
            });
        }
    }
}

template <class Ar>
int run(const Limb &p, const Ar &ar, const u64 *in, u64 *out, bool forward) {
    switch (ntt_n2(p.logn)) {
        case 7: row_pass<7>(p, ar, in, out, forward); return 0;
        case 8: row_pass<8>(p, ar, in, out, forward); return 0;
        case 9: row_pass<9>(p, ar, in, out, forward); return 0;
        default: return -1;
    }
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
template <class Ar>
static int col_run(const Limb &p, const Ar &ar, const u64 *in, u64 *out, bool forward) {
    // canonical residues enter an inverse as 2 units of 0.52 q (FP64)
    const int bound = forward ? (Ar::kFp ? 16 : 4) : (Ar::kFp ? 2 : 3);
    switch (ntt_n1(p.logn)) {
        case 6: col_pass<6>(p, ar, in, out, forward, bound); return 0;
        case 7: col_pass<7>(p, ar, in, out, forward, bound); return 0;
        case 8: col_pass<8>(p, ar, in, out, forward, bound); return 0;
        default: return -1;
    }
}

// A whole transform by column and row tiles: forward canonical coefficients to
// natural-order values, inverse back.
extern "C" int emu_fused_ntt(const uint64_t *in, uint64_t *out, uint64_t q, uint32_t logn, int forward) {
    if (logn < 13 || logn > 17 || q >= kLazyModulusBound) return -1;
    if (!host::negacyclic_root(q, 1ull << logn)) return -2;
    const Limb p(q, logn);
    std::vector<uint64_t> mid(1ull << logn);
    auto go = [&](const auto &ar) {
        int rc = forward ? col_run(p, ar, in, mid.data(), true) : run(p, ar, in, mid.data(), false);
        if (rc) return rc;
        return forward ? run(p, ar, mid.data(), out, true) : col_run(p, ar, mid.data(), out, false);
    };
    return p.fp ? go(RowFp{(double)q, 1.0 / (double)q}) : go(RowInt{q});
}

// shoup_lazy3 at y w mod q: the residue it returns (before any reduction)
extern "C" uint64_t emu_shoup_lazy3(uint64_t y, uint64_t w, uint64_t q) {
    return shoup_lazy3(y, w, host::shoup_quotient(w, q), q);
}
