// Fused NTT passes (gfx950): column passes that read a key switch's digits in
// the form it has them, and row passes that do its pointwise work between the
// forward and the inverse transform of one tile, so NTT-domain data never
// reaches HBM.  The tiles are in col_tile.hpp and row_tile.hpp.
#include "host_math.hpp"
#include "fused.hpp"
#include "fused_dev.hpp"
#include "ntt_pass.hpp"
#include "routes.hpp"
#include "col_tile.hpp"

namespace ck {

// ---- row products -------------------------------------------------------------

// psi^e for e < N is T[bitrev(e)], psi^(N + e) = -psi^e; the Shoup quotient of
// q - w is 2^64 - 1 - floor(w 2^64 / q) (w 2^64 / q is no integer).
__global__ __launch_bounds__(256) void k_row_products(const Tw *table, u64 q, u32 fp, u32 logn, void *out) {
    const u32 x = blockIdx.x * 256 + threadIdx.x, N = 1u << logn;
    if (x >= N) return;
    const u32 n2 = ntt_n2(logn), n1 = logn - n2;
    const u32 u = bitrev(x >> n2, n1), t = x & ((1u << n2) - 1);
    const u32 e = ((2 * u + 1) * t) & (2 * N - 1);
    const Tw w = table[bitrev(e & (N - 1), logn)];
    if (fp) {
        const double d = u64_as_f64(w.w);
        ((double *)out)[x] = e >= N ? (double)q - d : d;
    } else {
        ((Tw *)out)[x] = e >= N ? Tw{q - w.w, ~w.wq} : w;
    }
}

int build_row_products(hipStream_t s, const Tw *table, u64 q, bool fp, u32 logn, void *out) {
    const u32 N = 1u << logn;
    hipLaunchKernelGGL(k_row_products, dim3(N / 256), dim3(256), 0, s, table, q, fp ? 1u : 0u, logn, out);
    CK_HIP(hipGetLastError());
    return CKKS_OK;
}

bool fused_rows_apply(const ckks_rns_plan *plan) {
    if (plan->logn < 13 || plan->logn > 17) return false;
    for (u64 q : plan->moduli)
        if (q >= kLazyModulusBound) return false;
    return true;
}

// ---- column passes --------------------------------------------------------------

// One entry of a launch.  The inter-pass side is limb-major: limb transform
// limb * n_polys + poly.
struct ColEntry {
    const u64 *src;
    u64 *dst;
    const DevPrime *primes;
    u64 stride;       // elements between polynomials on the coefficient side
    u32 n_polys, n_limbs, logn, block_start;
    u32 kind, digits;  // ColKind; polynomials per ciphertext (lifts)
    u64 limit;         // digits: 2^(w-1)
    const ColBlock *blocks;
    const u64 *m;      // inverse: ColAdd operands
    const int64_t *err;
    u64 m_stride;
    u32 add;
    unsigned char order[kMaxOrder];  // limb_order
};

constexpr int kMaxColEntries = 16;

struct ColLaunch {
    ColEntry e[kMaxColEntries];
    u32 n, blocks;
};

template <class C>
__device__ __forceinline__ void col_read(u64 (&v)[C::M], const u64 *src, u32 n2, u32 tile, u32 tid, u32 kind) {
    const u32 o0 = C::template offset<0>(tile, n2, tid, 0) * 8;
    if (kind == kColInt8) {
        const int8_t *b = (const int8_t *)src;
#pragma unroll
        for (int i = 0; i < C::M; ++i) v[i] = (u64)(int64_t)(b + C::template step<0>(n2, i))[o0 / 8];
    } else if (kind == kColPlain) {
#pragma unroll
        for (int i = 0; i < C::M; ++i) v[i] = load_once_at(src + C::template step<0>(n2, i), o0);
    } else {
        // read once per target limb: not streamed
#pragma unroll
        for (int i = 0; i < C::M; ++i) v[i] = load_at(src + C::template step<0>(n2, i), o0);
    }
}

template <class C, class Ar>
__device__ __forceinline__ void col_blocks(u64 (&v)[C::M], const u64 *src, u64 N, const CK_CONST_AS ColBlock &blk,
                                           u32 limb, u32 n2, u32 tile, u32 tid, const CK_CONST_AS DevPrime &P) {
    typedef BlockSum<Ar::kFp> Sum;
    constexpr int W = 8;  // residues summed at a time: what their partial sums leave room for
    const u32 o0 = C::template offset<0>(tile, n2, tid, 0) * 8;
    const CK_CONST_AS u64 *row0 = const_table(blk.rows) + (u64)limb * kColTerms * 2;
    const u32 first = blk.first, terms = blk.terms, split = blk.split;
#pragma unroll
    for (int g = 0; g < C::M; g += W) {
        Sum s[W];
        u64 x[W];
        const CK_CONST_AS u64 *row = row0;
        const u64 *d = src + (u64)first * N;
#pragma unroll
        for (int i = 0; i < W; ++i) x[i] = load_at(d + C::template step<0>(n2, g + i), o0);
        u32 t = 0;
        if (split) {
#pragma unroll
            for (int i = 0; i < W; ++i) {
                s[i].add((x[i] & 0x3fffffffu) | kDigitBias, row[0], u64_as_f64(row[1]));
                s[i].add((x[i] >> 30) | kDigitBias, row[2], u64_as_f64(row[3]));
                if (i & 1) sched_fence();
            }
            t = 2;
        } else {
#pragma unroll
            for (int i = 0; i < W; ++i) s[i].add(x[i] | kDigitBias, row[0], u64_as_f64(row[1]));
            t = 1;
        }
#pragma unroll 1
        for (row += 2 * t; t < terms; ++t, row += 2) {
            d += N;
#pragma unroll
            for (int i = 0; i < W; ++i) x[i] = load_at(d + C::template step<0>(n2, g + i), o0);
            const u64 w = row[0];
            const double wp = u64_as_f64(row[1]);
#pragma unroll
            for (int i = 0; i < W; ++i) {
                s[i].add(x[i] | kDigitBias, w, wp);
                if ((i & 3) == 3) sched_fence();
            }
        }
#pragma unroll
        for (int i = 0; i < W; ++i) {
            v[g + i] = s[i].value(P.q);
            if (i & 1) sched_fence();
        }
    }
}

template <class C, bool BLOCK, class Ar>
__device__ __forceinline__ void col_forward(const ColEntry &e, const CK_CONST_AS DevPrime &P, const Ar &ar, u32 limb,
                                            u32 poly, u32 tile, u64 *lds) {
    const u32 tid = threadIdx.x, n2 = e.logn - C::K;
    const u64 N = (u64)1 << e.logn;
    const u64 *src = nullptr;
    u64 limit = 0;
    if (BLOCK) {
    } else if (e.kind == kColPlain) {
        src = e.src + poly * e.stride + limb * N;
    } else if (e.kind == kColInt8) {
        src = (const u64 *)((const int8_t *)e.src + poly * N);
    } else {
        // digit j of ciphertext ct, shared by every limb
        const u32 ct = poly / e.digits, j = poly % e.digits;
        src = e.src + ct * e.stride + j * N;
        limit = e.kind == kColResidue ? const_table(e.primes)[j].q : e.limit;
    }
    u64 v[C::M];
    int b[C::M];
    if (BLOCK) {
        const u32 ct = poly / e.digits, j = poly % e.digits;
        col_blocks<C, Ar>(v, e.src + ct * e.stride, N, const_table(e.blocks)[j], limb, n2, tile, tid, P);
    } else {
        col_read<C>(v, src, n2, tile, tid, e.kind);
        col_lift(v, e.kind, limit, ar, P);
    }
    C::set(b, Ar::kFp ? kColFpIn : kColIntIn);
    C::template fwd<0>(v, b, tid, P.fwd, ar);
    C::template put<0>(v, tid, lds);
    // on to the row pass: times psi^((2u+1) t)
    u64 *dst = e.dst + ((u64)limb * e.n_polys + poly) * N;
    const typename Ar::Z *z = (const typename Ar::Z *)P.zf;
    const u32 o1 = C::template offset<C::LAST>(tile, n2, tid, 0);
    typename Ar::Z zv[C::M];
    if (Ar::kFp) {
#pragma unroll
        for (int i = 0; i < C::M; ++i) zv[i] = load_z(z + C::template step<C::LAST>(n2, i), o1);
    }
    __syncthreads();
    C::template get<1>(v, tid, lds);
    C::level(b);
    C::template fwd<1>(v, b, tid, P.fwd, ar);
    if constexpr (C::LAST == 2) {
        __syncthreads();
        C::template put<1>(v, tid, lds);
        __syncthreads();
        C::template get<2>(v, tid, lds);
        C::level(b);
        C::template fwd<2>(v, b, tid, P.fwd, ar);
    }
#pragma unroll
    for (int i = 0; i < C::M; ++i) {
        const u32 st = C::template step<C::LAST>(n2, i);
        // 16-byte row products: a few in flight at a time
        if (!Ar::kFp) zv[i] = load_z(z + st, o1);
        store_once_at(dst + st, o1 * 8, ar.times(v[i], zv[i]));
        if (!Ar::kFp && (i & 3) == 3) sched_fence();
    }
}

template <class C, bool ADD, class Ar>
__device__ __forceinline__ void col_inverse(const ColEntry &e, const CK_CONST_AS DevPrime &P, const Ar &ar, u32 limb,
                                            u32 poly, u32 tile, u64 *lds) {
    const u32 tid = threadIdx.x, n2 = e.logn - C::K;
    const u64 N = (u64)1 << e.logn;
    const u64 *src = e.src + ((u64)limb * e.n_polys + poly) * N;
    u64 *dst = e.dst + poly * e.stride + limb * N;
    u64 v[C::M];
    int b[C::M];
    const typename Ar::Z *z = (const typename Ar::Z *)P.zi;
    const u32 o1 = C::template offset<C::LAST>(tile, n2, tid, 0);
#pragma unroll
    for (int i = 0; i < C::M; ++i) {
        const u32 st = C::template step<C::LAST>(n2, i);
        v[i] = load_once_at(src + st, o1 * 8);
    }
#pragma unroll
    for (int i = 0; i < C::M; ++i) {
        v[i] = ar.times(v[i], load_z(z + C::template step<C::LAST>(n2, i), o1));
        if (!Ar::kFp && (i & 3) == 3) sched_fence();
    }
    C::set(b, Ar::kZ);
    if constexpr (C::LAST == 2) {
        C::template inv<2>(v, b, tid, P.inv, ar);
        C::template put<2>(v, tid, lds);
        __syncthreads();
        C::template get<1>(v, tid, lds);
        C::level(b);
        __syncthreads();
    }
    C::template inv<1>(v, b, tid, P.inv, ar);
    C::template put<1>(v, tid, lds);
    __syncthreads();
    C::template get<0>(v, tid, lds);
    C::level(b);
    C::template inv<0>(v, b, tid, P.inv, ar);
    const u32 o0 = C::template offset<0>(tile, n2, tid, 0) * 8;
#pragma unroll
    for (int i = 0; i < C::M; ++i) {
        u64 r;
        if constexpr (Ar::kFp) {
            r = fp_residue(fp_mulmod(u64_as_f64(v[i]), P.ninv_d, P.ninv_p, ar.q), ar.q, ar.qinv);
        } else {
            r = shoup(v[i], P.ninv, P.ninv_q, ar.q);
        }
        if constexpr (ADD) {
            const u32 st = C::template step<0>(n2, i);
            const u64 m = load_once_at(e.m + poly * e.m_stride + limb * N + st, o0);
            if (e.add == kAddBody) {
                r = add_mod(m, r, P.q);
            } else {
                const int64_t x = (int64_t)load_at((const u64 *)e.err + poly * N + st, o0);
                const u64 mag = x < 0 ? 0 - (u64)x : (u64)x;
                u64 er = mag;
                if (mag >= P.q) er = barrett_reduce128(0, mag, Barrett{P.q, P.br_hi, P.br_lo});
                if (x < 0) er = neg_mod(er, P.q);
                r = sub_mod(add_mod(m, er, P.q), r, P.q);
            }
        }
        store_once_at(dst + C::template step<0>(n2, i), o0, r);
        if (!Ar::kFp && (i & 3) == 3) sched_fence();
    }
}

// Blocks of an entry.  Lifts: the limbs of one (polynomial, tile) follow each
// other on one XCD, which reads the shared input once into its L2.  Plain and
// inverse passes take four limbs of every polynomial at a time: the four
// limbs' row products stay in the XCDs' L2s over the batch (all limbs' do
// not), and heavy limbs still run beside light ones.
constexpr u32 kColGroup = 4;

// OTHER: kColBlock digits (forward) or ColAdd (inverse), which take more registers
template <bool FWD, bool OTHER, int B>
__global__ __launch_bounds__(4096 >> B, B == 3 || OTHER ? 4 : 5) void k_columns(ColLaunch l) {
    __shared__ u64 lds[4096];
    u32 di = 0;
    while (di + 1 < l.n && blockIdx.x >= l.e[di + 1].block_start) ++di;
    const ColEntry &e = l.e[di];
    const u32 b = blockIdx.x - e.block_start, lt = e.logn - 12, tiles = 1u << lt;
    u32 limb, poly, tile;
    if (FWD && e.kind != kColPlain && e.kind != kColInt8) {
        const u32 k = b >> 3, group = k / e.n_limbs * 8 + (b & 7);
        if (group >= e.n_polys * tiles) return;
        limb = k % e.n_limbs;
        poly = group >> lt;
        tile = group & (tiles - 1);
    } else {
        tile = b & (tiles - 1);
        const u32 x = b >> lt, per = kColGroup * e.n_polys, whole = e.n_limbs / kColGroup;
        const u32 grp = x / per < whole ? x / per : whole;
        const u32 width = grp < whole ? kColGroup : e.n_limbs % kColGroup, y = x - grp * per;
        poly = y / width;
        limb = grp * kColGroup + y % width;
    }
    if (e.n_limbs <= kMaxOrder) limb = e.order[limb];
    const CK_CONST_AS DevPrime &P = const_table(e.primes)[limb];
    const RowFp fp{P.qd, P.qinv};
    const RowInt in{P.q};
    switch (e.logn - ntt_n2(e.logn)) {
#define CK_COL(K1)                                                            \
    case K1: {                                                                \
        typedef ColTile<K1, B> C;                                             \
        if (FWD) {                                                            \
            if (P.fp) col_forward<C, OTHER>(e, P, fp, limb, poly, tile, lds);      \
            else col_forward<C, OTHER>(e, P, in, limb, poly, tile, lds);           \
        } else {                                                              \
            if (P.fp) col_inverse<C, OTHER>(e, P, fp, limb, poly, tile, lds);      \
            else col_inverse<C, OTHER>(e, P, in, limb, poly, tile, lds);           \
        }                                                                     \
        break;                                                                \
    }
        CK_COL(6)
        CK_COL(7)
        CK_COL(8)
#undef CK_COL
    }
}

// Tiles up to which a launch takes the 512-thread form (ColTile B = 3), where a
// CU has few waves to hide latencies in.  4 ciphertexts at N = 2^13 (208 and 208
// tiles): mixed-radix digits 18.7 -> 12.4 us, inverse 10.1 -> 8.2 us.  Above, the
// 16-residue form with its one exchange wins: inverse of 800 tiles 21.9 / 25.6 us,
// of 65536 tiles 1250 / 1667 us.
constexpr u32 kWideColumns = 512;
int launch_columns(ckks_context *ctx, const ColCall *calls, size_t count, bool forward) {
    if (count > (size_t)kMaxColEntries) return fail(CKKS_ERR_INVALID, "NTT batch holds at most 16 entries");
    ColLaunch l{}, lo{};  // lo: OTHER entries of k_columns
    for (size_t i = 0; i < count; ++i) {
        const ColCall &c = calls[i];
        ColLaunch &to = (forward ? c.kind == kColBlock : c.add != kAddNone) ? lo : l;
        if (c.n_polys == 0) continue;
        if (!fused_rows_apply(c.plan)) return fail(CKKS_ERR_UNSUPPORTED, "column passes: two-pass degrees, primes below 2^60");
        ColEntry e{};
        e.src = c.in;
        e.dst = c.out;
        e.primes = c.plan->d_primes;
        e.stride = c.stride;
        e.n_polys = (u32)c.n_polys;
        e.n_limbs = (u32)c.n_limbs;
        e.logn = c.plan->logn;
        e.block_start = to.blocks;
        e.kind = (u32)c.kind;
        e.digits = (u32)c.digits;
        e.limit = c.limit;
        e.blocks = c.blocks;
        e.m = c.m;
        e.err = c.e;
        e.m_stride = c.m_stride;
        e.add = (u32)c.add;
        limb_order(c.plan, c.n_limbs, e.order);
        to.e[to.n++] = e;
        const size_t groups = c.n_polys << (e.logn - 12);
        const size_t blocks = to.blocks + (forward && c.kind != kColPlain && c.kind != kColInt8 ? (groups + 7) / 8 * 8 : groups) * c.n_limbs;
        to.blocks = (u32)blocks;
        if (blocks >= (1ull << 31)) return fail(CKKS_ERR_INVALID, "NTT batch too large for one launch");
        ckks_execution_profile &pc = ctx->counts();
        (forward ? pc.ntt_forwards : pc.ntt_inverses) += c.n_polys;
        pc.ntt_limb_transforms += c.n_polys * c.n_limbs;
    }
    const auto launch = [&](auto fwd, auto other, const ColLaunch &c) {
        constexpr bool F = decltype(fwd)::value, O = decltype(other)::value;
        if (c.blocks == 0) return;
        if (c.blocks <= kWideColumns)
            hipLaunchKernelGGL((k_columns<F, O, 3>), dim3(c.blocks), dim3(512), 0, ctx->stream, c);
        else
            hipLaunchKernelGGL((k_columns<F, O, 4>), dim3(c.blocks), dim3(256), 0, ctx->stream, c);
    };
    if (forward) {
        launch(std::true_type(), std::false_type(), l);
        launch(std::true_type(), std::true_type(), lo);
    } else {
        launch(std::false_type(), std::false_type(), l);
        launch(std::false_type(), std::true_type(), lo);
    }
    CK_HIP(hipGetLastError());
    return CKKS_OK;
}

// ---- block order ----------------------------------------------------------------

// Workgroups (limb, tile, ciphertext).  Integer limbs cost two to three times
// an FP64 limb and are spread evenly (limb_order); blocks reach the 8 XCDs round-robin,
// and group (limb, tile) g runs on XCD g mod 8 with its ciphertexts one after
// another, so its key tile is read into one L2 and every XCD gets the same
// share of heavy limbs.
struct RowGrid {
    u32 n_cts, limbs, logn, groups;
    u32 tb;   // a tile is 2^tb residues
    u32 xcd;  // 0: ciphertexts of a group on consecutive blocks
    unsigned char order[kMaxOrder];
};

// half: tiles up to which they halve (routes.hpp)
static RowGrid row_grid(const ckks_rns_plan *plan, size_t limbs, size_t n_cts, bool xcd, size_t half = kHalfTiles) {
    RowGrid g{};
    g.n_cts = (u32)n_cts;
    g.limbs = (u32)limbs;
    g.logn = plan->logn;
    g.tb = limb_tiles(limbs, n_cts, plan->logn) <= half ? 11 : 12;
    g.groups = (u32)(limbs << (plan->logn - g.tb));
    g.xcd = xcd ? 1u : 0u;
    limb_order(plan, limbs, g.order);
    return g;
}

static u32 row_blocks(const RowGrid &g) { return g.xcd ? (g.groups + 7) / 8 * 8 * g.n_cts : g.groups * g.n_cts; }

struct RowBlock {
    u32 ct, limb, tile;
    bool idle;
};

__device__ __forceinline__ RowBlock row_block(const RowGrid &g, u32 b) {
    RowBlock r;
    u32 group;
    if (g.xcd) {
        const u32 l = b >> 3;
        group = l / g.n_cts * 8 + (b & 7);
        r.ct = l % g.n_cts;
    } else {
        group = b / g.n_cts;
        r.ct = b % g.n_cts;
    }
    r.idle = group >= g.groups;
    const u32 lt = g.logn - g.tb, pos = group >> lt;
    r.tile = group & ((1u << lt) - 1);
    r.limb = r.idle ? 0 : g.limbs <= kMaxOrder ? g.order[pos] : pos;
    return r;
}

// ---- key inner product ------------------------------------------------------------

struct RowMacArgs {
    RowMacJob e[kRowJobs];
    const DevPrime *primes;
    RowGrid grid;  // n_cts: of all jobs
    u32 dnum, count;
};

// An exchange writes one of two LDS buffers and reads it after the barrier; the
// buffer's previous readers passed the other exchange's barrier in between, so
// one barrier per exchange is enough, also from one transform to the next.
template <class R>
using RowLds = u64[R::LDS];

// geometry A (inter-pass) -> C (natural), bounds in b
template <class R, class Ar>
__device__ __forceinline__ void row_forward(u64 (&v)[8], int (&b)[8], u32 tid, const Tw *tw, RowLds<R> *lds,
                                            const Ar &ar) {
    typename R::LowTw low;
    R::template fwd<0>(v, b, tid, tw, low, ar);
    R::template put<0>(v, tid, lds[0]);
    __syncthreads();
    R::template get<1>(v, tid, lds[0]);
    R::level(b);
    R::template fwd<1>(v, b, tid, tw, low, ar);
    R::template put<1>(v, tid, lds[1]);
    low = R::low_twiddles(tw, tid);
    __syncthreads();
    R::template get<2>(v, tid, lds[1]);
    R::level(b);
#pragma unroll
    for (int x = 0; x < (1 << R::EX); ++x) R::fwd_group(v, b, x, low, ar);
}

template <class R, class Ar>
__device__ __forceinline__ void row_inverse(u64 (&v)[8], int (&b)[8], u32 tid, const Tw *tw, u64 *l0, u64 *l1,
                                            const Ar &ar) {
    const typename R::LowTw low = R::low_twiddles(tw, tid);
    R::template inv<2>(v, b, tid, tw, low, ar);
    R::template put<2>(v, tid, l0);
    __syncthreads();
    R::template get<1>(v, tid, l0);
    R::level(b);
    R::template inv<1>(v, b, tid, tw, low, ar);
    R::template put<1>(v, tid, l1);
    __syncthreads();
    R::template get<0>(v, tid, l1);
    R::level(b);
    R::template inv<0>(v, b, tid, tw, low, ar);
}

// NTT-domain entries of geometry C: register i sits bitrev(t) rows from the
// thread's first, the 2^EX columns of a thread adjacent and 16-byte aligned.
template <int L>
__device__ __forceinline__ void natural_read(u64 (&w)[8], const u64 *k, u32 n1, u32 nat0) {
    typedef RowTile<L> R;  // the same for every tile size
#pragma unroll
    for (int i = 0; i < 8; i += R::EX ? 2 : 1) {
        const u64 *at = k + (bitrev((u32)i >> R::EX, L) << n1) + (i & ((1 << R::EX) - 1));
        if constexpr (R::EX > 0) {
            const u64x2 p = load2_at(at, nat0);
            w[i] = p.x;
            w[i + 1] = p.y;
        } else {
            w[i] = load_at(at, nat0);
        }
    }
}

template <int L, int TB, class Ar, class Sum>
struct RowMacBody {
    typedef RowTile<L, TB> R;
    const RowMacArgs &a;
    const CK_CONST_AS DevPrime &P;
    const Ar ar;
    const Sum sum;
    RowLds<R> *lds;
    u32 tid;

    __device__ __forceinline__ void run(const RowBlock &blk) {
        const u32 logn = a.grid.logn, n1 = logn - L;
        const u64 N = (u64)1 << logn;
        const u32 off0 = R::internal_off(blk.tile, n1, tid, 0) * 8;
        const u32 nat0 = R::natural_off(blk.tile, n1, tid, 0) * 8;
        const u32 D = a.dnum;
        u32 job = 0;
        while (job + 1 < a.count && blk.ct >= a.e[job + 1].first) ++job;
        const RowMacJob &e = a.e[job];
        const u64 poly = (u64)blk.limb * e.n_cts + (blk.ct - e.first);
        const u64 *src = e.digits + poly * D * N;
        const u64 *kb = e.kb + (u64)blk.limb * N, *ka = e.ka + (u64)blk.limb * N;
        const u64 kstride = (u64)a.grid.limbs * N;
        typename Sum::S sb[8], sa[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) sb[i] = sa[i] = 0;
        typename R::LowTw low;
        u64 v[8], nx[8], wb[8], wa[8];
        int b[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) nx[i] = load_at(src + (i << (L - 3)), off0);
#pragma unroll 1
        for (u32 j = 0;; ++j) {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = nx[i];
            R::set(b, Ar::kZ);
            tid = opaque(tid);
            auto next = [&]() {
                src += N;
                if (j + 1 < D) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) nx[i] = load_at(src + (i << (L - 3)), off0);
                }
            };
            // the key entries and the next digit are on their way while the
            // stages run, each requested as late as registers allow
            natural_read<L>(wb, kb, n1, nat0);
            R::template fwd<0>(v, b, tid, P.fwd, low, ar);
            R::template put<0>(v, tid, lds[0]);
            next();
            __syncthreads();
            R::template get<1>(v, tid, lds[0]);
            R::level(b);
            R::template fwd<1>(v, b, tid, P.fwd, low, ar);
            R::template put<1>(v, tid, lds[1]);
            natural_read<L>(wa, ka, n1, nat0);
            low = R::low_twiddles(P.fwd, tid);
            __syncthreads();
            R::template get<2>(v, tid, lds[1]);
            R::level(b);
#pragma unroll
            for (int x = 0; x < (1 << R::EX); ++x) {
                R::fwd_group(v, b, x, low, ar);
#pragma unroll
                for (int i = x; i < 8; i += 1 << R::EX) {
                    sum.mac(sb[i], v[i], wb[i]);
                    sum.mac(sa[i], v[i], wa[i]);
                    if (!Ar::kFp) sched_fence();
                }
                sched_fence();
            }
            kb += kstride;
            ka += kstride;
            if (j + 1 == D) break;
            if (Sum::full(j)) {
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    sb[i] = sum.reduced(sb[i]);
                    sa[i] = sum.reduced(sa[i]);
                }
            }
        }
        tid = opaque(tid);
        u64 *out = e.out + poly * 2 * N;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = sum.total(c ? sa[i] : sb[i]);
            R::set(b, Sum::kIn);
            row_inverse<R>(v, b, tid, P.inv, lds[0], lds[1], ar);
#pragma unroll
            for (int i = 0; i < 8; ++i) *(u64 *)((char *)(out + c * N + (i << (L - 3))) + off0) = v[i];
        }
    }
};

template <int L, int TB>
__global__ __launch_bounds__(1 << (TB - 3), TB == 11 ? 2 : 4) void k_row_mac(RowMacArgs a) {
    typedef RowTile<L, TB> R;
    __shared__ __align__(16) u64 lds[2][R::LDS];
    const RowBlock blk = row_block(a.grid, blockIdx.x);
    if (blk.idle) return;
    const CK_CONST_AS DevPrime &P = const_table(a.primes)[blk.limb];
    if (P.fp)
        RowMacBody<L, TB, RowFp, SumFp>{a, P, RowFp{P.qd, P.qinv}, SumFp{P.qd, P.qinv}, lds, threadIdx.x}.run(blk);
    else
        RowMacBody<L, TB, RowInt, SumInt>{a, P, RowInt{P.q}, SumInt(P.q, P.br_hi, P.br_lo), lds, threadIdx.x}.run(blk);
}

int launch_row_mac(ckks_context *ctx, RowMac &m) {
    if (!fused_rows_apply(m.plan)) return fail(CKKS_ERR_UNSUPPORTED, "fused row passes: 2^13 <= N <= 2^17, primes below 2^60");
    if (m.count == 0 || m.count > kRowJobs) return fail(CKKS_ERR_INVALID, "1..16 key switches a launch");
    RowMacArgs a{};
    size_t n_cts = 0;
    for (size_t i = 0; i < m.count; ++i) {
        m.e[i].first = (u32)n_cts;
        a.e[i] = m.e[i];
        n_cts += m.e[i].n_cts;
    }
    a.count = (u32)m.count;
    a.primes = m.plan->d_primes;
    a.grid = row_grid(m.plan, m.limbs, n_cts, m.xcd_order, row_mac_half_tiles(ntt_n2(m.plan->logn)));
    a.dnum = (u32)m.dnum;
    if ((u64)m.limbs * n_cts << (m.plan->logn - 12) >= (1ull << 30))
        return fail(CKKS_ERR_INVALID, "key-switch batch too large for one launch");
    const dim3 g(row_blocks(a.grid)), t(1u << (a.grid.tb - 3));
    switch (ntt_n2(m.plan->logn) * 2 + a.grid.tb - 11) {
#define CK_ROW(L)                                                                                          \
    case L * 2: hipLaunchKernelGGL((k_row_mac<L, 11>), g, t, 0, ctx->stream, a); break;                    \
    case L * 2 + 1: hipLaunchKernelGGL((k_row_mac<L, 12>), g, t, 0, ctx->stream, a); break;
        CK_ROW(7) CK_ROW(8) CK_ROW(9)
#undef CK_ROW
    }
    CK_HIP(hipGetLastError());
    return CKKS_OK;
}

// ---- products of polynomials -------------------------------------------------------

// Products for operands the forward pass left lazy.  factor() brings one of
// them into the range the product wants (FP64: half a q; integer: 4 q, so that
// T = 16 q 4 q < 2^126 and the Montgomery product stays below 5 q).
__device__ __forceinline__ void row_factor(u64 (&v)[8], int (&)[8], const RowFp &ar) {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = f64_as_u64(fp_reduce(u64_as_f64(v[i]), ar.q, ar.qinv));
}
__device__ __forceinline__ void row_factor(u64 (&v)[8], int (&b)[8], const RowInt &ar) {
#pragma unroll
    for (int i = 0; i < 8; ++i) ar.reduce_to(v[i], b[i], 4);
}
// s += y w: w from row_factor
__device__ __forceinline__ void row_mac(double &s, u64 y, u64 w, const SumFp &sum) {
    s += fp_mulmod_q(u64_as_f64(y), u64_as_f64(w), sum.q, sum.qinv);
}
__device__ __forceinline__ void row_mac(u64 &s, u64 y, u64 w, const SumInt &sum) { sum.mac(s, y, w); }

struct RowMulArgs {
    u64 *x;        // inter-pass [limb][poly][N]
    const u64 *y;  // inter-pass [limb][N], or null
    const u64 *w;  // natural [limb][N] at w + (poly / share) w_stride
    u64 w_stride;
    u32 share;
    const DevPrime *primes;
    RowGrid grid;  // n_cts: polynomials
};

// Forward, product, inverse of one tile: against separate passes this leaves
// out two or three passes over the data and as many launches.  With the column
// passes (memory-bound like this one: 16 bytes a residue) a plaintext product
// of 16 ciphertexts and its rescale take 224 us at N = 2^15, 13 limbs (308 us
// with separate passes), an encryption of 8 polynomials there 118 us (184 us).
template <int L, bool INTER, class R, class Ar, class Sum>
__device__ __forceinline__ void row_mul_tile(const RowMulArgs &a, const CK_CONST_AS DevPrime &P, const Ar &ar,
                                             const Sum &sum, RowLds<R> *lds, const RowBlock &blk) {
    const u32 tid = threadIdx.x, logn = a.grid.logn, n1 = logn - L;
    const u64 N = (u64)1 << logn;
    const u32 off0 = R::internal_off(blk.tile, n1, tid, 0) * 8;
    u64 *x = a.x + ((u64)blk.limb * a.grid.n_cts + blk.ct) * N;
    u64 v[8], w[8];
    int b[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = load_at(x + (i << (L - 3)), off0);
    if constexpr (INTER) {
        const u64 *y = a.y + (u64)blk.limb * N;
#pragma unroll
        for (int i = 0; i < 8; ++i) w[i] = load_at(y + (i << (L - 3)), off0);
        R::set(b, Ar::kZ);
        row_forward<R>(w, b, tid, P.fwd, lds, ar);
        row_factor(w, b, ar);
    } else {
        const u64 *k = a.w + blk.ct / a.share * a.w_stride + (u64)blk.limb * N;
        natural_read<L>(w, k, n1, R::natural_off(blk.tile, n1, tid, 0) * 8);
    }
    R::set(b, Ar::kZ);
    row_forward<R>(v, b, tid, P.fwd, lds, ar);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        typename Sum::S s = 0;
        if constexpr (INTER) row_mac(s, v[i], w[i], sum);
        else sum.mac(s, v[i], w[i]);
        v[i] = sum.total(s);
    }
    R::set(b, Sum::kIn);
    row_inverse<R>(v, b, tid, P.inv, lds[0], lds[1], ar);
#pragma unroll
    for (int i = 0; i < 8; ++i) *(u64 *)((char *)(x + (i << (L - 3))) + off0) = v[i];
}

template <int L, int TB, bool INTER>
__global__ __launch_bounds__(1 << (TB - 3), TB == 11 ? 2 : 4) void k_row_mul(RowMulArgs a) {
    typedef RowTile<L, TB> R;
    __shared__ __align__(16) u64 lds[2][R::LDS];
    const RowBlock blk = row_block(a.grid, blockIdx.x);
    if (blk.idle) return;
    const CK_CONST_AS DevPrime &P = const_table(a.primes)[blk.limb];
    if (P.fp)
        row_mul_tile<L, INTER, R>(a, P, RowFp{P.qd, P.qinv}, SumFp{P.qd, P.qinv}, lds, blk);
    else
        row_mul_tile<L, INTER, R>(a, P, RowInt{P.q}, SumInt(P.q, P.br_hi, P.br_lo), lds, blk);
}

int launch_row_mul(ckks_context *ctx, const RowMul &m) {
    if (!fused_rows_apply(m.plan)) return fail(CKKS_ERR_UNSUPPORTED, "fused row passes: 2^13 <= N <= 2^17, primes below 2^60");
    RowMulArgs a{};
    a.x = m.x;
    a.y = m.y;
    a.w = m.w;
    a.w_stride = m.w_stride;
    a.share = (u32)m.share;
    a.primes = m.plan->d_primes;
    a.grid = row_grid(m.plan, m.limbs, m.n_polys, true);
    if ((u64)m.limbs * m.n_polys << (m.plan->logn - 12) >= (1ull << 30))
        return fail(CKKS_ERR_INVALID, "NTT batch too large for one launch");
    const dim3 g(row_blocks(a.grid)), t(1u << (a.grid.tb - 3));
    switch ((ntt_n2(m.plan->logn) * 2 + a.grid.tb - 11) * 2 + (m.y ? 1 : 0)) {
#define CK_ROW(L, TB, X)                                                                                       \
    case (L * 2 + TB - 11) * 2 + X: hipLaunchKernelGGL((k_row_mul<L, TB, X>), g, t, 0, ctx->stream, a); break;
#define CK_ROWS(L) CK_ROW(L, 11, 0) CK_ROW(L, 11, 1) CK_ROW(L, 12, 0) CK_ROW(L, 12, 1)
        CK_ROWS(7) CK_ROWS(8) CK_ROWS(9)
#undef CK_ROWS
#undef CK_ROW
    }
    CK_HIP(hipGetLastError());
    return CKKS_OK;
}

struct RowTensorArgs {
    u64 *x[4];  // inter-pass b0, a0, b1, a1, each [limb][ct][N]
    const DevPrime *primes;
    RowGrid grid;
};

// Four forward row passes, the products and three inverse passes of one tile;
// b0 and a0 stay in registers as factors while b1 and a1 are transformed.
template <int L, class R, class Ar, class Sum>
__device__ __forceinline__ void row_tensor_tile(const RowTensorArgs &a, const CK_CONST_AS DevPrime &P, const Ar &ar,
                                                const Sum &sum, RowLds<R> *lds, const RowBlock &blk) {
    u32 tid = threadIdx.x;
    const u32 n1 = a.grid.logn - L;
    const u64 base = ((u64)blk.limb * a.grid.n_cts + blk.ct) << a.grid.logn;
    const u32 off0 = R::internal_off(blk.tile, n1, tid, 0) * 8;
    u64 f[2][8], v[8];  // b0 and a0 as factors
    typename Sum::S c[3][8];
    int b[8];
#pragma unroll
    for (int p = 0; p < 2; ++p) {
#pragma unroll
        for (int i = 0; i < 8; ++i) f[p][i] = load_at(a.x[p] + base + (i << (L - 3)), off0);
        R::set(b, Ar::kZ);
        tid = opaque(tid);
        row_forward<R>(f[p], b, tid, P.fwd, lds, ar);
        row_factor(f[p], b, ar);
    }
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int i = 0; i < 8; ++i) c[k][i] = 0;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = load_at(a.x[2 + p] + base + (i << (L - 3)), off0);
        R::set(b, Ar::kZ);
        tid = opaque(tid);
        row_forward<R>(v, b, tid, P.fwd, lds, ar);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            row_mac(c[p][i], v[i], f[0][i], sum);
            row_mac(c[p + 1][i], v[i], f[1][i], sum);
            sched_fence();
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = sum.total(c[k][i]);
        R::set(b, Sum::kIn);
        tid = opaque(tid);
        row_inverse<R>(v, b, tid, P.inv, lds[0], lds[1], ar);
#pragma unroll
        for (int i = 0; i < 8; ++i) *(u64 *)((char *)(a.x[k] + base + (i << (L - 3))) + off0) = v[i];
    }
}

template <int L, int TB>
__global__ __launch_bounds__(1 << (TB - 3), TB == 11 ? 2 : 4) void k_row_tensor(RowTensorArgs a) {
    typedef RowTile<L, TB> R;
    __shared__ __align__(16) u64 lds[2][R::LDS];
    const RowBlock blk = row_block(a.grid, blockIdx.x);
    if (blk.idle) return;
    const CK_CONST_AS DevPrime &P = const_table(a.primes)[blk.limb];
    if (P.fp)
        row_tensor_tile<L, R>(a, P, RowFp{P.qd, P.qinv}, SumFp{P.qd, P.qinv}, lds, blk);
    else
        row_tensor_tile<L, R>(a, P, RowInt{P.q}, SumInt(P.q, P.br_hi, P.br_lo), lds, blk);
}

int launch_row_tensor(ckks_context *ctx, const ckks_rns_plan *plan, u64 *const x[4], size_t n_cts, size_t limbs) {
    if (!fused_rows_apply(plan)) return fail(CKKS_ERR_UNSUPPORTED, "fused row passes: 2^13 <= N <= 2^17, primes below 2^60");
    RowTensorArgs a{};
    for (int p = 0; p < 4; ++p) a.x[p] = x[p];
    a.primes = plan->d_primes;
    a.grid = row_grid(plan, limbs, n_cts, true);
    if ((u64)limbs * n_cts << (plan->logn - 12) >= (1ull << 30))
        return fail(CKKS_ERR_INVALID, "NTT batch too large for one launch");
    const dim3 g(row_blocks(a.grid)), t(1u << (a.grid.tb - 3));
    switch (ntt_n2(plan->logn) * 2 + a.grid.tb - 11) {
#define CK_ROW(L)                                                                                          \
    case L * 2: hipLaunchKernelGGL((k_row_tensor<L, 11>), g, t, 0, ctx->stream, a); break;                    \
    case L * 2 + 1: hipLaunchKernelGGL((k_row_tensor<L, 12>), g, t, 0, ctx->stream, a); break;
        CK_ROW(7) CK_ROW(8) CK_ROW(9)
#undef CK_ROW
    }
    CK_HIP(hipGetLastError());
    return CKKS_OK;
}

// ---- hoisted rotations -------------------------------------------------------------

struct RowRotateArgs {
    const u64 *digits, *bhat;
    const DevPrime *primes;
    RowRotation e[kRowRotations];
    RowGrid grid;  // n_cts: rotations of every ciphertext, the exponent fastest
    u32 count, dnum, q_limbs;
};

// v + a canonical x; `b` grows by kCanonical
__device__ __forceinline__ u64 plus(u64 v, u64 x, const RowFp &) { return f64_as_u64(u64_as_f64(v) + small_to_f64(x)); }
__device__ __forceinline__ u64 plus(u64 v, u64 x, const RowInt &) { return v + x; }

// Key products of the digits of one tile, sigma_k and the inverse row pass.
// Evaluation point n = T N1 + u of the result is point ((2n + 1) k - 1) / 2 of
// the sums, so sigma_k takes row u to row u' as a whole ((2u' + 1) k = 2u + 1
// mod 2 N1: the store goes to another 2^L-residue run) and permutes within it,
// T -> T k^-1 + c(u): one more exchange through LDS.  The permuted sums never
// reach HBM.  4 rotations of 16 ciphertexts at N = 2^16, 25 + 7 limbs, dnum 3:
// 1.58 ms, where the products (0.81 ms) and a permuting first inverse pass
// (1.23 ms) took two launches.  What bounds it is the entries each workgroup
// reads from L2 (keys alone: 1.18 ms without them); sharing them between two
// ciphertexts of a workgroup took the registers that it saved in loads
// (1.55 ms with spills), one workgroup per sum 1.83 ms.
template <int L, class R, class Ar, class Sum>
__device__ __forceinline__ void row_rotate_tile(const RowRotateArgs &a, const CK_CONST_AS DevPrime &P, const Ar &ar,
                                                const Sum &sum, RowLds<R> *lds, const RowBlock &blk) {
    constexpr int EX = R::EX, CL = R::CL;
    constexpr int kCanonical = Ar::kFp ? 2 : 1;
    u32 tid = threadIdx.x;
    const u32 logn = a.grid.logn, n1 = logn - L;
    const u64 N = (u64)1 << logn, stride = (u64)a.grid.limbs * N;
    const u32 ct = blk.ct / a.count;
    const RowRotation &e = a.e[blk.ct % a.count];
    const u32 nat0 = R::natural_off(blk.tile, n1, tid, 0) * 8;
    const u64 *src = a.digits + (u64)ct * a.dnum * stride + (u64)blk.limb * N;
    const u64 *kb = e.kb + (u64)blk.limb * N, *ka = e.ka + (u64)blk.limb * N;
    typename Sum::S sb[8], sa[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) sb[i] = sa[i] = 0;
    u64 v[8], w[8];
#pragma unroll 1
    for (u32 j = 0;; ++j) {
        u64 wa[8];
        natural_read<L>(v, src, n1, nat0);
        natural_read<L>(w, kb, n1, nat0);
        natural_read<L>(wa, ka, n1, nat0);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const u64 y = sum_input(v[i], ar);
            sum.mac(sb[i], y, w[i]);
            sum.mac(sa[i], y, wa[i]);
            if (!Ar::kFp || (i & 1)) sched_fence();
        }
        if (j + 1 == a.dnum) break;
        if (Sum::full(j)) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                sb[i] = sum.reduced(sb[i]);
                sa[i] = sum.reduced(sa[i]);
            }
        }
        src += stride;
        kb += stride;
        ka += stride;
    }
    const u32 mask2 = (2u << logn) - 1, rows = (1u << L) - 1;
    u64 *out = e.out + ((u64)blk.limb * (a.grid.n_cts / a.count) + ct) * 2 * N;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        int b[8], bound = Sum::kIn;
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = sum.total(c ? sa[i] : sb[i]);
        if (e.tb) {
            natural_read<L>(w, (c ? e.ta : e.tb) + (u64)blk.limb * N, n1, nat0);
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = plus(v[i], w[i], ar);
        }
        bound += kCanonical;
        if (c == 0 && a.bhat && blk.limb < a.q_limbs) {
            natural_read<L>(w, a.bhat + ((u64)ct * a.q_limbs + blk.limb) * N, n1, nat0);
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = plus(v[i], w[i], ar);
        }
        if (c == 0) bound += kCanonical;
        // sigma_k: the two sums take turns with the buffers, so that no put
        // meets a get of the same buffer without a barrier between them
        tid = opaque(tid);
        {
            const u32 T0 = bitrev(R::t_of(2, tid, 0), L) * e.kinv;
            const u32 u0 = (blk.tile << CL) + R::col_of(2, tid, 0);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const u32 col = (u32)i & ((1u << EX) - 1), x = bitrev((u32)i >> EX, L);
                const u32 carry = (((2 * (u0 + col) + 1) * e.kinv) & mask2) >> (n1 + 1);
                const u32 t = bitrev((T0 + x * e.kinv + carry) & rows, L);
                const u32 at = R::slot((t << CL) | (R::col_of(2, tid, 0) + col));
                CK_BOUNDS(at, (u32)R::LDS);
                lds[c][at] = v[i];
            }
        }
        __syncthreads();
        R::template get<2>(v, tid, lds[c]);
        R::set(b, bound);
        row_inverse<R>(v, b, tid, P.inv, lds[1 - c], lds[c], ar);
        const u32 u = (blk.tile << CL) + R::col_of(0, tid, 0);
        const u32 to = (((2 * u + 1) * e.kinv) & ((2u << n1) - 1)) >> 1;
        const u32 off = ((bitrev(to, n1) << L) + R::t_of(0, tid, 0)) * 8;
#pragma unroll
        for (int i = 0; i < 8; ++i) *(u64 *)((char *)(out + c * N + (i << (L - 3))) + off) = v[i];
    }
}

template <int L, int TB>
__global__ __launch_bounds__(1 << (TB - 3), TB == 11 ? 2 : 4) void k_row_rotate(RowRotateArgs a) {
    typedef RowTile<L, TB> R;
    __shared__ __align__(16) u64 lds[2][R::LDS];
    const RowBlock blk = row_block(a.grid, blockIdx.x);
    if (blk.idle) return;
    const CK_CONST_AS DevPrime &P = const_table(a.primes)[blk.limb];
    if (P.fp)
        row_rotate_tile<L, R>(a, P, RowFp{P.qd, P.qinv}, SumFp{P.qd, P.qinv}, lds, blk);
    else
        row_rotate_tile<L, R>(a, P, RowInt{P.q}, SumInt(P.q, P.br_hi, P.br_lo), lds, blk);
}

int launch_row_rotate(ckks_context *ctx, const RowRotate &r) {
    if (!fused_rows_apply(r.plan)) return fail(CKKS_ERR_UNSUPPORTED, "fused row passes: 2^13 <= N <= 2^17, primes below 2^60");
    if (r.count == 0 || r.count > (size_t)kRowRotations) return fail(CKKS_ERR_INVALID, "1..16 exponents a launch");
    RowRotateArgs a{};
    a.digits = r.digits;
    a.bhat = r.bhat;
    a.primes = r.plan->d_primes;
    for (size_t i = 0; i < r.count; ++i) a.e[i] = r.e[i];
    a.count = (u32)r.count;
    a.dnum = (u32)r.dnum;
    a.q_limbs = (u32)r.q_limbs;
    a.grid = row_grid(r.plan, r.limbs, r.n_cts * r.count, true, row_rotate_half_tiles(r.dnum, ntt_n2(r.plan->logn)));
    if ((u64)r.limbs * r.n_cts * r.count << (r.plan->logn - 12) >= (1ull << 30))
        return fail(CKKS_ERR_INVALID, "NTT batch too large for one launch");
    const dim3 g(row_blocks(a.grid)), t(1u << (a.grid.tb - 3));
    switch (ntt_n2(r.plan->logn) * 2 + a.grid.tb - 11) {
#define CK_ROW(L)                                                                                          \
    case L * 2: hipLaunchKernelGGL((k_row_rotate<L, 11>), g, t, 0, ctx->stream, a); break;                    \
    case L * 2 + 1: hipLaunchKernelGGL((k_row_rotate<L, 12>), g, t, 0, ctx->stream, a); break;
        CK_ROW(7) CK_ROW(8) CK_ROW(9)
#undef CK_ROW
    }
    CK_HIP(hipGetLastError());
    return CKKS_OK;
}

}  // namespace ck
