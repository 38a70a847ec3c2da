// eo_pipelined.hip -- the pipelined iterations of the even-odd solvers, FP32 for mixed precision
// and FP64: one launch per CG iteration on S^T S, S the Schur complement on the even sites
// (evenodd.hip).
//
// CG with the residual norm recurrence of D'Azevedo, Eijkhout and Romine (LAPACK Working Note 56,
// 1993): with rho = |r|^2, mu = <p, Ap>, nu = |Ap|^2, alpha_k = rho_k / mu_k and
// <r_k, Ap_k> = mu_k, rho_{k+1} = alpha_k^2 nu_k - rho_k, so beta_{k+1} is known before r_{k+1}
// exists and the x, r updates move into the next operator application.
//
// One block owns a TT x TX tile of the full lattice (TT, TX even) and produces Ap on the tile's
// even sites.  It works on the tile with a 4-site halo, (TT+8) x (TX+8) sites: entry (row, k)
// holds the even and the odd site of columns 2k and 2k+1, at the same index of the half-lattice
// vectors.  A thread keeps the same M0 entries through all stages, so that both sites' own values
// stay in registers and a hop reads three of its four neighbours from LDS (the fourth is the
// entry's other site); each stage fills the parity it produces on a halo one site smaller:
//   0: r' = r - alpha Ap, p' = r' + beta p on even sites, 4-site halo (own sites also written
//      out, and the x update)
//   1: U = K p' / d on odd sites, 3-site halo          (= A_o^-1 K_oe p')
//   2: v = d p' - K U on even sites, 2-site halo        (= S p', overwrites p')
//   3: W = H v / d on odd sites, 1-site halo            (overwrites U)
//   4: Ap = d v - H W on the tile's even sites          (= S^T S p')
// The block partials are (mu, nu) = (|v|^2, |Ap|^2) and (rho', 0), rho' the exact |r'|^2 that
// re-anchors the recurrence every iteration.  Ap ping-pongs between two buffers and the directions
// rotate through three: blocks read the old ones on their halo while others write the new ones.
//
// Bytes per even site and launch in FP32: 88 B (even) and 120 B (odd launches, which also update
// x_s); twice that in FP64.
#include <algorithm>
#include <type_traits>

#include "pipelined.hpp"

namespace ycn {

struct EoPfArgs {
    int Nt, Nh, Vh, nNoise;
    double r, d0, g;
    int tilesX, tilesPerSys, xcdRemap;
    float invNt, invNh;
};

// minus the hop K (DAG) or H of an entry's site from the other parity's array N: the time
// neighbours at i +- K, one space neighbour at io and the other `own`, which is the left one
// where sg = 1 and the right one where sg = -1
template <typename R, bool DAG, bool WR1, typename Lds>
__device__ __forceinline__ Sp<R> eo_pf_hop(R r, const Lds &N, int i, int K, int io, Sp<R> own, R sg, R sf, R sb) {
    using V2 = typename Vec2<R>::T;
    const R h = (R)0.5, sTb = DAG ? sf : sb, sTf = DAG ? sb : sf;
    const int iTb = DAG ? i + K : i - K, iTf = DAG ? i - K : i + K;
    const Sp<R> o = N.get(io);
    const V2 tb0 = N.s0(iTb), tf1 = N.s1(iTf);
    const R a = DAG ? -sg : sg;   // (back - forward) = a (own - other)
    Sp<R> q;
    if constexpr (WR1) {
        q.a.x = sTb * tb0.x + h * ((own.a.x + o.a.x) + a * (own.b.x - o.b.x));
        q.a.y = sTb * tb0.y + h * ((own.a.y + o.a.y) + a * (own.b.y - o.b.y));
        q.b.x = sTf * tf1.x + h * ((own.b.x + o.b.x) + a * (own.a.x - o.a.x));
        q.b.y = sTf * tf1.y + h * ((own.b.y + o.b.y) + a * (own.a.y - o.a.y));
    } else {
        const V2 tb1 = N.s1(iTb), tf0 = N.s0(iTf);
        const R hp = h * (r + (R)1), hm = h * (r - (R)1), hr = h * r, ha = h * a;
        const R ap = hp * sTb, am = hm * sTf, bm = hm * sTb, bp = hp * sTf;
        q.a.x = ap * tb0.x + am * tf0.x + hr * (own.a.x + o.a.x) + ha * (own.b.x - o.b.x);
        q.a.y = ap * tb0.y + am * tf0.y + hr * (own.a.y + o.a.y) + ha * (own.b.y - o.b.y);
        q.b.x = bm * tb1.x + bp * tf1.x + hr * (own.b.x + o.b.x) + ha * (own.a.x - o.a.x);
        q.b.y = bm * tb1.y + bp * tf1.y + hr * (own.b.y + o.b.y) + ha * (own.a.y - o.a.y);
    }
    return q;
}
template <typename R>
__device__ __forceinline__ Sp<R> scale(R s, Sp<R> v) {
    return {mk2<R>(s * v.a.x, s * v.a.y), mk2<R>(s * v.b.x, s * v.b.y)};
}

// Launch idx of a chunk.  PERSIST: the grid holds as many blocks as are resident, each walks the
// tiles blockIdx.x, blockIdx.x + gridDim.x, ... and loads the next tile's vectors while it runs
// stages 1-4 of the current one; one partial per block.
// finMode 0: alpha and beta from the state, a finalize launch follows.  1: the launch finalizes
// its predecessor in its prologue (pf_prologue): every block sums prevPart in the same order and
// derives the same alpha, beta and stop; launch 0 of a chunk starts from the state, a closing
// launch finalizes the last.  2: timing, neither pausing nor writing the state.
// RM, where r_{idx-1} comes from:
//   1: r itself, with alpha = 0 (launch 0, after the setup or a reliable update put it there);
//   2: rebuilt as p_{idx-1} - beta_{idx-1} p_{idx-2}, the relation that formed p_{idx-1}; r then
//      carries p_{idx-2}.  The rounding of the rebuild is a few eps |p| against the eps |r| of a
//      stored r (|p| is a few |r| in CG).
// XM, the x update: 0: none (an even launch); 2: the odd launch after it adds both terms,
// alpha_{idx-2} p_{idx-2} + alpha p_{idx-1}.  A system that stops after an odd number of launches
// (at the iteration cap) leaves a term to the reliable update or the close.
// Block 0 records the alpha, beta of the launch in the state as ab[idx & 1] for the next one.
template <typename R, int TT, int TX, int NT, bool PERSIST, bool WR1, int XM, int RM>
__global__ void __launch_bounds__(NT)
k_eo_pf(EoPfArgs A, const typename Vec2<R>::T *__restrict__ phi, CgState *st,
        const typename Vec2<R>::T *__restrict__ r, const typename Vec2<R>::T *__restrict__ Ap_in,
        const typename Vec2<R>::T *__restrict__ pold, typename Vec2<R>::T *__restrict__ pnew,
        typename Vec2<R>::T *__restrict__ Ap, typename Vec2<R>::T *__restrict__ xs, double2 *__restrict__ part,
        int finMode, int idx, const double2 *__restrict__ prevPart, int *active) {
    using V2 = typename Vec2<R>::T;
    constexpr int H = TT + 8, K = (TX + 8) / 2, N = H * K, M0 = (N + NT - 1) / NT;
    constexpr bool FP64 = sizeof(R) == 8;
    __shared__ SpLds<R, N> E;
    __shared__ SpLds<R, N - 2 * K> O;   // rows 1 .. H - 2, shifted down by one row
    __shared__ double red[3 * NT / kWave], bc[2];
    __shared__ int pause;
    const int sys = blockIdx.y;
    const PfHead hd = pf_head(st[sys]);
    const double2 prev = RM == 2 ? st[sys].ab[(idx - 1) & 1] : make_double2(0.0, 0.0);
    PfParts<NT> parts;
    if (finMode && idx) parts.load(prevPart + 2 * (size_t)sys * gridDim.x, (int)gridDim.x);
    if (hd.done) return;
    const unsigned Vh = (unsigned)A.Vh;
    const size_t off = (size_t)sys * 2 * Vh;
    r += off;
    Ap_in += off;
    pold += off;
    pnew += off;
    Ap += off;
    xs += off;
    phi += (size_t)(sys / A.nNoise) * Vh;

    // an entry's place: 1 = even site within the 2-site halo, 2 = its even site is the tile's own,
    // 4 = odd site within the 3-site halo, 8 = within the 1-site halo; 16, 32: hops across the
    // time boundary, forward and backward; 64: odd row
    int at_[M0];
#pragma unroll
    for (int u = 0; u < M0; ++u) {
        const int w = threadIdx.x + u * NT, row = w / K, k = w - row * K, odd = row & 1;
        const int ce = 2 * k + odd, co = 2 * k + 1 - odd;
        auto in = [&](int col, int h) {
            return row >= 4 - h && row < 4 + TT + h && col >= 4 - h && col < 4 + TX + h;
        };
        at_[u] = w >= N ? 0 : (in(ce, 2) ? 1 : 0) | (in(ce, 0) ? 2 : 0) | (in(co, 3) ? 4 : 0) | (in(co, 1) ? 8 : 0) |
                                  (odd ? 64 : 0);
    }
    struct Regs {
        Sp<R> a[M0], p[M0], q[M0], x[M0];
        V2 f[M0];
        unsigned j[M0];
        int edge[M0];
    } G;
    auto load = [&](int tile) {
        if (A.xcdRemap) tile = (tile % 8) * (A.tilesPerSys / 8) + tile / 8;   // bands of tiles per XCD
        const int ty = tile / A.tilesX, t0 = ty * TT, h0 = (tile - ty * A.tilesX) * (TX / 2);
#pragma unroll
        for (int u = 0; u < M0; ++u) {
            const int w = threadIdx.x + u * NT;
            if (w < N) {
                const int row = w / K, k = w - row * K;
                const int gt = wrapf(t0 - 4 + row, A.Nt, A.invNt), gh = wrapf(h0 - 2 + k, A.Nh, A.invNh);
                const unsigned j = (unsigned)(gt * A.Nh + gh);
                G.j[u] = j;
                G.edge[u] = (gt == A.Nt - 1 ? 16 : 0) | (gt == 0 ? 32 : 0);
                G.a[u] = load_sp<R>(r, Vh, j);
                G.p[u] = load_sp<R>(pold, Vh, j);
                if (RM == 2) G.q[u] = load_sp<R>(Ap_in, Vh, j);
                if (XM != 0 && (at_[u] & 2)) G.x[u] = load_sp<R>(xs, Vh, j);
                G.f[u] = at(phi, j);
            }
        }
    };
    int tile = blockIdx.x;
    load(tile);
    double alphaD, betaD;
    if constexpr (FP64) {
        if (!p64_prologue<NT>(st, hd, sys, idx, finMode, parts, prevPart, active, red, bc, &pause, alphaD, betaD))
            return;
    } else {
        if (!pf_prologue<NT>(st, hd, sys, idx, finMode, parts, prevPart, part, active, red, bc, &pause, alphaD, betaD))
            return;
    }
    if (blockIdx.x == 0 && threadIdx.x == 0) st[sys].ab[idx & 1] = make_double2(RM == 1 ? 0.0 : alphaD, betaD);
    const R alpha = (R)alphaD, beta = (R)betaD, alphaPrev = (R)prev.x, betaPrev = (R)prev.y;
    const R wr = (R)A.r;

    double rho = 0.0, mu = 0.0, nu = 0.0;
    while (true) {
        Sp<R> e[M0], o[M0];   // the entry's even and odd site
        R de[M0], inv[M0];    // d of the even site, 1 / d of the odd one
        R sg[M0], sf[M0], sb[M0];   // signs: row parity, hops across the time boundary
        unsigned j[M0];
        int place[M0];
#pragma unroll
        for (int u = 0; u < M0; ++u) {
            const int w = threadIdx.x + u * NT;
            place[u] = 0;
            if (w < N) {
                place[u] = at_[u] | G.edge[u];
                j[u] = G.j[u];
                const bool odd = place[u] & 64;
                sg[u] = odd ? (R)-1 : (R)1;
                sf[u] = place[u] & 16 ? (R)-1 : (R)1;
                sb[u] = place[u] & 32 ? (R)-1 : (R)1;
                de[u] = (R)A.d0 + (R)A.g * (odd ? G.f[u].y : G.f[u].x);
                inv[u] = (R)1 / ((R)A.d0 + (R)A.g * (odd ? G.f[u].x : G.f[u].y));
                Sp<R> a = G.a[u];
                if (RM == 2) a = axpy<R>(axpy<R>(G.p[u], -betaPrev, a), -alpha, G.q[u]);
                e[u] = axpy<R>(a, beta, G.p[u]);
                E.set(w, e[u]);
                if (place[u] & 2) {
                    rho += sq(a);
                    store_sp<R>(pnew, Vh, j[u], e[u]);
                    if (XM == 2)
                        store_sp<R>(xs, Vh, j[u], axpy<R>(axpy<R>(G.x[u], alphaPrev, G.a[u]), alpha, G.p[u]));
                }
            }
        }
        __syncthreads();
        if (PERSIST && tile + (int)gridDim.x < A.tilesPerSys) load(tile + (int)gridDim.x);
        // odd sites: the entry's even site is the left neighbour in an even row
        auto odd_stage = [&](auto dag, int bit) {
#pragma unroll
            for (int u = 0; u < M0; ++u)
                if (place[u] & bit) {
                    const int w = threadIdx.x + u * NT;
                    o[u] = scale<R>(-inv[u],
                                    eo_pf_hop<R, decltype(dag)::value, WR1>(wr, E, w, K, place[u] & 64 ? w - 1 : w + 1,
                                                                            e[u], sg[u], sf[u], sb[u]));
                    O.set(w - K, o[u]);
                }
        };
        // even sites: the entry's odd site is the right neighbour in an even row
        auto even_site = [&](auto dag, int u) {
            const int w = threadIdx.x + u * NT - K;
            return axpy<R>(eo_pf_hop<R, decltype(dag)::value, WR1>(wr, O, w, K, place[u] & 64 ? w + 1 : w - 1, o[u],
                                                                   -sg[u], sf[u], sb[u]),
                           de[u], e[u]);
        };
        odd_stage(std::true_type(), 4);
        __syncthreads();
#pragma unroll
        for (int u = 0; u < M0; ++u)
            if (place[u] & 1) {
                e[u] = even_site(std::true_type(), u);
                E.set(threadIdx.x + u * NT, e[u]);
                if (place[u] & 2) mu += sq(e[u]);
            }
        __syncthreads();
        odd_stage(std::false_type(), 8);
        __syncthreads();
#pragma unroll
        for (int u = 0; u < M0; ++u)
            if (place[u] & 2) {
                const Sp<R> v = even_site(std::false_type(), u);
                store_sp<R>(Ap, Vh, j[u], v);
                nu += sq(v);
            }
        if (!PERSIST) break;
        tile += (int)gridDim.x;
        if (tile >= A.tilesPerSys) break;   // (stage 0 writes E only, which stage 4 does not read)
    }
    store_pf_partials<NT>(part + 2 * ((size_t)sys * gridDim.x + blockIdx.x), mu, nu, rho, red);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// form 0: launch 0 of a phase (r read), 1: odd launches, 2: even ones; returns the block partials
// per system
template <typename R, int TT, int TX, int NT>
static int launch_tt(const Ctx &c, int nsys, const EoPfLaunch<R> &b) {
    using V2 = typename Vec2<R>::T;
    EoPfArgs A;
    A.Nt = c.p.Nt;
    A.Nh = c.p.Nx / 2;
    A.Vh = c.V / 2;
    A.nNoise = c.nNoise;
    A.r = c.p.r;
    A.d0 = 2.0 * c.p.r + c.p.M;
    A.g = c.p.g;
    A.tilesX = c.p.Nx / TX;
    A.tilesPerSys = (c.p.Nt / TT) * A.tilesX;
    A.xcdRemap = A.tilesPerSys % 8 == 0 ? 1 : 0;
    A.invNt = 1.0f / (float)A.Nt;
    A.invNh = 1.0f / (float)A.Nh;
    int grid = A.tilesPerSys;
    auto go = [&](auto persistTag, auto wrTag) {
        constexpr bool P = decltype(persistTag)::value, W1 = decltype(wrTag)::value;
        using K = decltype(&k_eo_pf<R, TT, TX, NT, P, W1, 0, 1>);
        static const K ks[3] = {&k_eo_pf<R, TT, TX, NT, P, W1, 0, 1>, &k_eo_pf<R, TT, TX, NT, P, W1, 2, 2>,
                                &k_eo_pf<R, TT, TX, NT, P, W1, 0, 2>};
        if (P) {
            static const int resident = resident_blocks(ks, NT);
            grid = persistent_grid(resident, A.tilesPerSys);
        }
        hipLaunchKernelGGL(ks[b.form], dim3(grid, nsys), dim3(NT), 0, c.stream, A,
                           reinterpret_cast<const V2 *>(b.phi), c.cg_d, b.r, b.Ap_in, b.pold, b.pnew, b.Ap, b.x, b.part,
                           b.finMode, b.idx, b.prevPart, c.active);
    };
    const bool w1 = c.p.r == 1.0;
    constexpr bool persistent = std::is_same<R, float>::value &&
                                (TT * TX == 256 || TT * TX == 512) && TT >= 8;   // 8x32, 16x16, 16x32, 8x64
    if constexpr (persistent) {
        if (b.persist) {
            w1 ? go(std::true_type(), std::true_type()) : go(std::true_type(), std::false_type());
            return grid;
        }
    }
    w1 ? go(std::false_type(), std::true_type()) : go(std::false_type(), std::false_type());
    return grid;
}

// Block sizes: the entries of the tile with its halo, TT + 8 rows of (TX + 8) / 2, spread over
// threads with few idle ones.  What bounds an iteration, measured per launch pair's average:
//   256 x 256 FP32, 8x32 tiles of one entry per thread: 5.0 us, latency (launch, the prologue's
//     sums, one load, four stages, the block's sums); 7.2 in the stage-indexed kernel before.
//   1024 x 1024 FP32: 13.3 us for 54 MB (6.6 us at the 8.2 TB/s of a cache-resident copy) with
//     64x64 and 32x128 tiles, which leave one block per compute unit, a quarter of the work in the
//     halo and 256 partials for the prologue; 15.7 with 16x32 on a persistent grid, 16.3 with 16x64;
//     18.5 before.  About 4 us are vector instructions, 1 the prologue, 1 the launch.
//   1024 x 1024 FP64: 23.3 us for 109 MB with 16x32 tiles of two entries per thread (several
//     blocks per compute unit, one loading while another works), 24.7 with one entry, 26.4 32x32.
//   512 x 512 FP64: 7.9 us with 32x32 tiles and 832 threads, 8.3 with 448, 8.6 with 16x32.
int launch_eo_pf32(const Ctx &c, int TT, int TX, int nsys, const EoPfLaunch<float> &b) {
    switch (TT * 1000 + TX) {
    case 8032: return launch_tt<float, 8, 32, 320>(c, nsys, b);
    case 16032: return launch_tt<float, 16, 32, 256>(c, nsys, b);
    case 8064: return launch_tt<float, 8, 64, 320>(c, nsys, b);
    case 16016: return launch_tt<float, 16, 16, 320>(c, nsys, b);
    case 4064: return launch_tt<float, 4, 64, 448>(c, nsys, b);
    case 2032: return launch_tt<float, 2, 32, 256>(c, nsys, b);
    case 32032: return launch_tt<float, 32, 32, 448>(c, nsys, b);
    case 64064: return launch_tt<float, 64, 64, 704>(c, nsys, b);
    case 32128: return launch_tt<float, 32, 128, 704>(c, nsys, b);
    default: return launch_tt<float, 16, 64, 448>(c, nsys, b);
    }
}
int launch_eo_pf64(const Ctx &c, int TT, int TX, int nsys, const EoPfLaunch<double> &b) {
    switch (TT * 1000 + TX) {
    case 8032: return launch_tt<double, 8, 32, 320>(c, nsys, b);
    case 16032: return launch_tt<double, 16, 32, 256>(c, nsys, b);
    case 16016: return launch_tt<double, 16, 16, 320>(c, nsys, b);
    case 4032: return launch_tt<double, 4, 32, 256>(c, nsys, b);
    case 2032: return launch_tt<double, 2, 32, 256>(c, nsys, b);
    case 4016: return launch_tt<double, 4, 16, 192>(c, nsys, b);
    default: return launch_tt<double, 32, 32, 832>(c, nsys, b);
    }
}

}  // namespace ycn
