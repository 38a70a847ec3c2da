// plain.hip -- the pipelined iterations of the plain solvers on D^dag D or D D^dag (packed real
// spinors), FP32 for mixed precision and FP64: one launch per CG iteration.
//
// The iteration is the even-odd one's (k_eo_pf in eo_pipelined.hip): CG with the residual
// norm recurrence of D'Azevedo, Eijkhout and Romine (LAPACK Working Note 56, 1993), so that one
// reduction per iteration suffices and the x and r updates move into the next application of
// the operator; r rebuilt from the directions after launch 0 of a chunk, x (x_s) updated by every
// other launch for both; the finalize in the next launch's prologue or a launch of its own.
// In FP32, per site and launch it reads p_{k-2} (or r), Ap, p and phi and writes p and Ap, and
// every other launch updates x_s: 84 and 116 B, against 4 x 16 + 4 and 6 x 16 B in four launches
// (operator, alpha, update, beta) before.  FP64: twice that, against 328 B in four launches.
//
// What bounds it: at 512 x 512 in FP32 the vectors stay in the caches and a launch is latency,
// its chain of partial sums, loads, two stencil stages and a reduction.  At 1024 x 1024 in FP64
// it moves 210 MB per launch out of the 256 MB last-level cache; an iteration takes 40 us there
// against 68 us for the four launches, 35 without A p in memory (k_pl_rc).
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "cg_fused.hpp"
#include "pipelined.hpp"

namespace ycn {

constexpr int kFcgNT = 448;   // of k_fcg_op: one entry of the tile with its halo per thread

struct PlArgs {
    int Nt, Nx, V, nNoise;
    double r, d0, g;
    int tilesX, tilesPerSys, xcdRemap;
};

// v times d minus the hop of D (DAG = false) or D^dag at array entry i of N (rows of W)
template <typename R, bool DAG, bool WR1, typename Lds>
__device__ __forceinline__ Sp<R> pl_dirac(R r, const Lds &N, int i, int W, R sf, R sb, R d, Sp<R> v) {
    using V2 = typename Vec2<R>::T;
    const R h = (R)0.5, sTb = DAG ? sf : sb, sTf = DAG ? sb : sf;
    const int iTb = DAG ? i + W : i - W, iTf = DAG ? i - W : i + W;
    const Sp<R> xf = N.get(DAG ? i - 1 : i + 1), xb = N.get(DAG ? i + 1 : i - 1);
    const V2 tb0 = N.s0(iTb), tf1 = N.s1(iTf);
    Sp<R> o;
    if constexpr (WR1) {
        o.a.x = sTb * tb0.x + h * ((xf.a.x + xb.a.x) + (xb.b.x - xf.b.x));
        o.a.y = sTb * tb0.y + h * ((xf.a.y + xb.a.y) + (xb.b.y - xf.b.y));
        o.b.x = sTf * tf1.x + h * ((xf.b.x + xb.b.x) + (xb.a.x - xf.a.x));
        o.b.y = sTf * tf1.y + h * ((xf.b.y + xb.b.y) + (xb.a.y - xf.a.y));
    } else {
        const V2 tb1 = N.s1(iTb), tf0 = N.s0(iTf);
        const R hp = h * (r + (R)1), hm = h * (r - (R)1), hr = h * r;
        const R ap = hp * sTb, am = hm * sTf, bm = hm * sTb, bp = hp * sTf;
        o.a.x = ap * tb0.x + am * tf0.x + hr * (xf.a.x + xb.a.x) + h * (xb.b.x - xf.b.x);
        o.a.y = ap * tb0.y + am * tf0.y + hr * (xf.a.y + xb.a.y) + h * (xb.b.y - xf.b.y);
        o.b.x = bm * tb1.x + bp * tf1.x + hr * (xf.b.x + xb.b.x) + h * (xb.a.x - xf.a.x);
        o.b.y = bm * tb1.y + bp * tf1.y + hr * (xf.b.y + xb.b.y) + h * (xb.a.y - xf.a.y);
    }
    return {mk2<R>(d * v.a.x - o.a.x, d * v.a.y - o.a.y), mk2<R>(d * v.b.x - o.b.x, d * v.b.y - o.b.y)};
}

// One launch of the iteration.  XM, RM, idx and finMode as in k_eo_pf; FIRST forms
// (XM 0, RM 1) read r and skip its update, alpha being 0.  A block owns a TT x TX tile (cut
// off at the lattice's edges); a thread keeps the same M0 entries of the tile with its 2-site
// halo through all stages, so that an entry's own values stay in registers.  FP64 keeps one
// array in LDS, for p and then for D p, with a barrier more, so that three blocks of 32 x 32
// sites fit a compute unit instead of one.
template <typename R, int TT, int TX, int NT, bool DAG1, bool WR1, int XM, int RM>
__global__ void __launch_bounds__(NT)
k_pl_pf(PlArgs A, const R *__restrict__ phi, CgState *st, const typename Vec2<R>::T *__restrict__ r,
        const typename Vec2<R>::T *__restrict__ Ap_in, const typename Vec2<R>::T *__restrict__ pold,
        typename Vec2<R>::T *__restrict__ pnew, typename Vec2<R>::T *__restrict__ Ap,
        typename Vec2<R>::T *__restrict__ xs, double2 *__restrict__ part, int finMode, int idx,
        const double2 *__restrict__ prevPart, int *active) {
    constexpr int H = TT + 4, W = TX + 4, N = H * W, M0 = (N + NT - 1) / NT;
    constexpr bool FP64 = sizeof(R) == 8;
    __shared__ SpLds<R, N> P;
    __shared__ SpLds<R, FP64 ? 1 : N> Q32;
    __shared__ double red[3 * NT / kWave], bc[2];
    __shared__ int pause;
    const int sys = blockIdx.y;
    const PfHead hd = pf_head(st[sys]);
    const double2 prev = RM == 2 ? st[sys].ab[(idx - 1) & 1] : make_double2(0.0, 0.0);
    PfParts<NT> parts;
    if (finMode && idx) parts.load(prevPart + 2 * (size_t)sys * gridDim.x, (int)gridDim.x);
    if (hd.done) return;
    const unsigned V = (unsigned)A.V;
    const size_t off = (size_t)sys * 2 * V;
    r += off;
    Ap_in += off;
    pold += off;
    pnew += off;
    Ap += off;
    xs += off;
    const R *ph = phi + (size_t)(sys / A.nNoise) * V;
    int tile = blockIdx.x;   // contiguous bands of tiles per XCD
    if (A.xcdRemap) tile = (tile % 8) * (A.tilesPerSys / 8) + tile / 8;
    const int ty = tile / A.tilesX, t0 = ty * TT, x0 = (tile - ty * A.tilesX) * TX;
    const int rowEnd = min(TT, A.Nt - t0) + 2, colEnd = min(TX, A.Nx - x0) + 2;

    // an entry's place: 1 = within the 1-site halo, 2 = the tile's own; 4, 8: the hops across
    // the time boundary, forward and backward
    Sp<R> a[M0], p[M0], q[M0], xv[M0];
    R d[M0];
    unsigned gs[M0];
    int at_[M0];
#pragma unroll
    for (int u = 0; u < M0; ++u) {
        const int i = threadIdx.x + u * NT;
        at_[u] = 0;
        if (i < N) {
            const int row = i / W, col = i - row * W;
            const int gt = wrapi(t0 - 2 + row, A.Nt), gx = wrapi(x0 - 2 + col, A.Nx);
            gs[u] = (unsigned)(gt * A.Nx + gx);
            const bool in1 = row >= 1 && row < H - 1 && col >= 1 && col < W - 1;
            const bool in2 = row >= 2 && row < rowEnd && col >= 2 && col < colEnd;
            at_[u] = (in1 ? 1 : 0) | (in2 ? 2 : 0) | (gt == A.Nt - 1 ? 4 : 0) | (gt == 0 ? 8 : 0);
            a[u] = load_sp<R>(r, V, gs[u]);
            p[u] = load_sp<R>(pold, V, gs[u]);
            if (RM == 2) q[u] = load_sp<R>(Ap_in, V, gs[u]);
            if (XM != 0 && in2) xv[u] = load_sp<R>(xs, V, gs[u]);
            d[u] = at(ph, gs[u]);
        }
    }
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
#pragma unroll
    for (int u = 0; u < M0; ++u) {
        const int i = threadIdx.x + u * NT;
        if (i < N) {
            d[u] = (R)A.d0 + (R)A.g * d[u];
            const Sp<R> p2 = a[u];
            if (RM == 2) a[u] = axpy<R>(axpy<R>(p[u], -betaPrev, a[u]), -alpha, q[u]);
            if (at_[u] & 2) {
                rho += sq(a[u]);
                if (XM == 2) store_sp<R>(xs, V, gs[u], axpy<R>(axpy<R>(xv[u], alphaPrev, p2), alpha, p[u]));
            }
            p[u] = axpy<R>(a[u], beta, p[u]);
            P.set(i, p[u]);
            if (at_[u] & 2) store_sp<R>(pnew, V, gs[u], p[u]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < M0; ++u)
        if (at_[u] & 1) {
            const int i = threadIdx.x + u * NT;
            q[u] = pl_dirac<R, DAG1, WR1>(wr, P, i, W, at_[u] & 4 ? (R)-1 : (R)1, at_[u] & 8 ? (R)-1 : (R)1, d[u],
                                          p[u]);
            if constexpr (!FP64) Q32.set(i, q[u]);
            if (at_[u] & 2) mu += sq(q[u]);
        }
    if constexpr (FP64) {
        __syncthreads();
#pragma unroll
        for (int u = 0; u < M0; ++u)
            if (at_[u] & 1) P.set(threadIdx.x + u * NT, q[u]);
    }
    __syncthreads();
    auto second = [&](const auto &Q) {
#pragma unroll
        for (int u = 0; u < M0; ++u)
            if (at_[u] & 2) {
                const int i = threadIdx.x + u * NT;
                const Sp<R> o = pl_dirac<R, !DAG1, WR1>(wr, Q, i, W, at_[u] & 4 ? (R)-1 : (R)1,
                                                        at_[u] & 8 ? (R)-1 : (R)1, d[u], q[u]);
                store_sp<R>(Ap, V, gs[u], o);
                nu += sq(o);
            }
    };
    if constexpr (FP64)
        second(P);
    else
        second(Q32);
    store_pf_partials<NT>(part + 2 * ((size_t)sys * gridDim.x + blockIdx.x), mu, nu, rho, red);
}

// The same launch (after the first of a phase) without A p in memory: p_{idx-1} is read with a
// 4-site halo and A p_{idx-1} computed again, by the same operations that gave its alpha, on the
// 2-site halo.  FP64 on lattices that fill the chip is bound by the last-level cache and has vector
// instructions to spare: per site and launch p_{idx-2}, p_{idx-1}, p and phi (104 B) and every
// other launch x (64 B more), against 168 and 232 B.  One array in LDS, two barriers per stage.
// Per iteration, 1024 x 1024 in a solve: 35 us (16x32 tiles, 512 threads) against 38, for 136 MB
// against 202; 512 x 512: 10.4 (32x32, 832 threads) against 11.4; at 256 x 256 the longer chain
// costs more than the traffic, 6.4 against 5.6.
template <typename R, int TT, int TX, int NT, bool DAG1, bool WR1, int XM>
__global__ void __launch_bounds__(NT)
k_pl_rc(PlArgs A, const R *__restrict__ phi, CgState *st, const typename Vec2<R>::T *__restrict__ pprev,
        const typename Vec2<R>::T *__restrict__ pold, typename Vec2<R>::T *__restrict__ pnew,
        typename Vec2<R>::T *__restrict__ xs, double2 *__restrict__ part, int finMode, int idx,
        const double2 *__restrict__ prevPart, int *active) {
    constexpr int H = TT + 8, W = TX + 8, N = H * W, M0 = (N + NT - 1) / NT;
    __shared__ SpLds<R, N> P;
    __shared__ double red[3 * NT / kWave], bc[2];
    __shared__ int pause;
    const int sys = blockIdx.y;
    const PfHead hd = pf_head(st[sys]);
    const double2 prev = st[sys].ab[(idx - 1) & 1];
    PfParts<NT> parts;
    if (finMode && idx) parts.load(prevPart + 2 * (size_t)sys * gridDim.x, (int)gridDim.x);
    if (hd.done) return;
    const unsigned V = (unsigned)A.V;
    const size_t off = (size_t)sys * 2 * V;
    pprev += off;
    pold += off;
    pnew += off;
    xs += off;
    const R *ph = phi + (size_t)(sys / A.nNoise) * V;
    int tile = blockIdx.x;   // contiguous bands of tiles per XCD
    if (A.xcdRemap) tile = (tile % 8) * (A.tilesPerSys / 8) + tile / 8;
    const int ty = tile / A.tilesX, t0 = ty * TT, x0 = (tile - ty * A.tilesX) * TX;
    const int rowEnd = min(TT, A.Nt - t0) + 4, colEnd = min(TX, A.Nx - x0) + 4;

    // an entry's place: 1 = the tile's own; 2, 16, 32 = within the 1-, 2-, 3-site halo; 4, 8: the
    // hops across the time boundary, forward and backward
    Sp<R> p[M0], q[M0], x[M0];
    R d[M0];
    unsigned g[M0];
    int place[M0];
#pragma unroll
    for (int u = 0; u < M0; ++u) {
        const int i = threadIdx.x + u * NT;
        place[u] = 0;
        if (i < N) {
            const int row = i / W, col = i - row * W;
            const int gt = wrapi(t0 - 4 + row, A.Nt), gx = wrapi(x0 - 4 + col, A.Nx);
            g[u] = (unsigned)(gt * A.Nx + gx);
            auto in = [&](int h) { return row >= h && row < H - h && col >= h && col < W - h; };
            const bool own = row >= 4 && row < rowEnd && col >= 4 && col < colEnd;
            place[u] = (own ? 1 : 0) | (in(3) ? 2 : 0) | (in(2) ? 16 : 0) | (in(1) ? 32 : 0) |
                       (gt == A.Nt - 1 ? 4 : 0) | (gt == 0 ? 8 : 0);
            p[u] = load_sp<R>(pold, V, g[u]);
            if (in(2)) q[u] = load_sp<R>(pprev, V, g[u]);
            if (XM != 0 && own) x[u] = load_sp<R>(xs, V, g[u]);
            d[u] = at(ph, g[u]);
        }
    }
    double alphaD, betaD;
    if (!p64_prologue<NT>(st, hd, sys, idx, finMode, parts, prevPart, active, red, bc, &pause, alphaD, betaD)) return;
    if (blockIdx.x == 0 && threadIdx.x == 0) st[sys].ab[idx & 1] = make_double2(alphaD, betaD);
    const R alpha = (R)alphaD, beta = (R)betaD, alphaPrev = (R)prev.x, betaPrev = (R)prev.y;
    const R wr = (R)A.r;
    auto dirac = [&](auto dag, int u, Sp<R> v) {
        return pl_dirac<R, decltype(dag)::value, WR1>(wr, P, threadIdx.x + u * NT, W, place[u] & 4 ? (R)-1 : (R)1,
                                                      place[u] & 8 ? (R)-1 : (R)1, d[u], v);
    };
    using First = std::integral_constant<bool, DAG1>;
    using Second = std::integral_constant<bool, !DAG1>;
    // v of the entries at `bit` into the array, once every thread has read what it holds
    auto put = [&](int bit, const Sp<R> (&v)[M0]) {
        __syncthreads();
#pragma unroll
        for (int u = 0; u < M0; ++u)
            if (place[u] & bit) P.set(threadIdx.x + u * NT, v[u]);
        __syncthreads();
    };

    double rho = 0.0, mu = 0.0, nu = 0.0;
#pragma unroll
    for (int u = 0; u < M0; ++u) {
        const int i = threadIdx.x + u * NT;
        if (i < N) {
            d[u] = (R)A.d0 + (R)A.g * d[u];
            P.set(i, p[u]);
            if (place[u] & 16) {
                if (XM == 2 && (place[u] & 1))
                    store_sp<R>(xs, V, g[u], axpy<R>(axpy<R>(x[u], alphaPrev, q[u]), alpha, p[u]));
                q[u] = axpy<R>(p[u], -betaPrev, q[u]);   // r_{idx-1}
            }
        }
    }
    __syncthreads();
    Sp<R> v[M0];
#pragma unroll
    for (int u = 0; u < M0; ++u)
        if (place[u] & 32) v[u] = dirac(First(), u, p[u]);
    put(32, v);
#pragma unroll
    for (int u = 0; u < M0; ++u)
        if (place[u] & 16) {
            const Sp<R> r = axpy<R>(q[u], -alpha, dirac(Second(), u, v[u]));
            p[u] = axpy<R>(r, beta, p[u]);
            if (place[u] & 1) {
                rho += sq(r);
                store_sp<R>(pnew, V, g[u], p[u]);
            }
        }
    put(16, p);
#pragma unroll
    for (int u = 0; u < M0; ++u)
        if (place[u] & 2) {
            v[u] = dirac(First(), u, p[u]);
            if (place[u] & 1) mu += sq(v[u]);
        }
    put(2, v);
#pragma unroll
    for (int u = 0; u < M0; ++u)
        if (place[u] & 1) nu += sq(dirac(Second(), u, v[u]));
    store_pf_partials<NT>(part + 2 * ((size_t)sys * gridDim.x + blockIdx.x), mu, nu, rho, red);
}

// ---------------------------------------------------------------------------
// flexible CG: the operator's launch
// ---------------------------------------------------------------------------
// Iteration i of a chunk of the flexible solver (Polak-Ribiere form, Notay, SIAM J. Sci. Comput. 22
// (2000)) is two launches: this one, p' = z + beta p and Ap, and the network's (k_cnn_fused), which
// takes alpha, updates x_s and r and makes the next z.  Each finalizes the other in its prologue.
// From iteration i - 1's <z, r'>, <z, Ap> and |r'|^2 every block derives the same
// beta = <z, r' - r> / <z_old, r> = -alpha <z, Ap> / rz_old and the same pause (at the stop or the
// drop after an even number of iterations, at the cap; a reliable update follows).  Block 0 records
// rz in ab[i & 1].y for the network's launch, or the pause.
struct FcgStep {
    double beta, rz;
    bool off, pause;
};
__device__ __forceinline__ FcgStep fcg_decide(const Pf3 &s, double2 prev, int iter, const PfHead &S) {
    FcgStep d;
    d.off = !isfinite(s.mu) || !isfinite(s.nu);   // switches the network off
    d.beta = d.off || !(prev.y > 0.0) ? 0.0 : -prev.x * s.nu / prev.y;
    d.rz = d.off ? prev.y : s.mu;
    const bool stop = !(sqrt(s.rho) > S.stop) || s.rho < kReliableDrop * kReliableDrop * S.rrRel;
    d.pause = iter >= S.maxIter || (stop && !(iter & 1));
    return d;
}
// the state after iteration number `iter`, for the reliable update; rhoPrev: |r|^2 before it
__device__ __forceinline__ void fcg_commit(CgState &S, const Pf3 &s, double2 prev, const FcgStep &d, int iter,
                                           int *active) {
    S.iter = iter;
    S.rr = s.rho;
    S.alpha = make_double2(prev.x, 0.0);
    S.rz_prev = prev.y;
    S.rz = d.rz;
    if (d.off) S.precOff = 1;
    if (d.pause) {
        S.done = 1;
        atomicSub(active, 1);
    }
}

// A block owns a 16 x 16 tile of one packed spinor: the system's (FL = 1), or one flavour's complex
// spinor (FL = 2: D keeps flavours and is real, so its two planes are like a packed spinor's:
// grid.y = system and flavour).
template <bool WR1, int FL>
__global__ void __launch_bounds__(kFcgNT)
k_fcg_op(PlArgs A, const float *__restrict__ phi, CgState *st, const float2 *__restrict__ z,
         const float2 *__restrict__ pold, float2 *__restrict__ pnew, float2 *__restrict__ Ap,
         double *__restrict__ part, int idx, const double2 *__restrict__ cnnPart, int nbCnn, int *active) {
    constexpr int TT = 16, TX = 16, NT = kFcgNT, H = TT + 4, W = TX + 4, N = H * W, M0 = (N + NT - 1) / NT;
    __shared__ SpLds<float, N> P, Q;
    __shared__ double red[3 * NT / kWave], bc[1];
    __shared__ int pause;
    const int sys = blockIdx.y / FL;
    const PfHead hd = pf_head(st[sys]);
    const double rz0 = st[sys].rz;
    const double2 prev = st[sys].ab[(idx - 1) & 1];
    PfParts<NT> parts;
    const double2 *const pp = cnnPart + 2 * (size_t)sys * nbCnn;
    if (idx) parts.load(pp, nbCnn);
    if (hd.done) return;
    const unsigned V = (unsigned)A.V;
    const size_t off = (size_t)blockIdx.y * 2 * V;
    z += off;
    pold += off;
    pnew += off;
    Ap += off;
    const float *ph = phi + (size_t)(sys / A.nNoise) * V;
    int tile = blockIdx.x;
    if (A.xcdRemap) tile = (tile % 8) * (A.tilesPerSys / 8) + tile / 8;
    const int ty = tile / A.tilesX, t0 = ty * TT, x0 = (tile - ty * A.tilesX) * TX;
    Sp<float> p[M0], q[M0];
    float d[M0];
    unsigned g[M0];
    int place[M0];   // as in k_pl_pf
#pragma unroll
    for (int u = 0; u < M0; ++u) {
        const int i = threadIdx.x + u * NT;
        place[u] = 0;
        if (i < N) {
            const int row = i / W, col = i - row * W;
            const int gt = wrapi(t0 - 2 + row, A.Nt), gx = wrapi(x0 - 2 + col, A.Nx);
            g[u] = (unsigned)(gt * A.Nx + gx);
            const bool in1 = row >= 1 && row < H - 1 && col >= 1 && col < W - 1;
            const bool in2 = row >= 2 && row < H - 2 && col >= 2 && col < W - 2;
            place[u] = (in1 ? 1 : 0) | (in2 ? 2 : 0) | (gt == A.Nt - 1 ? 4 : 0) | (gt == 0 ? 8 : 0);
            q[u] = load_sp<float>(z, V, g[u]);
            p[u] = load_sp<float>(pold, V, g[u]);
            d[u] = at(ph, g[u]);
        }
    }
    double betaD = hd.beta, rz = rz0;
    if (idx) {
        const Pf3 s = parts.sum(pp, nbCnn, red);
        if (threadIdx.x == 0) {
            const FcgStep f = fcg_decide(s, prev, hd.iter0 + idx, hd);
            bc[0] = f.beta;
            pause = f.pause;
            rz = f.rz;
            if (blockIdx.x == 0 && blockIdx.y % FL == 0) {
                if (f.pause)
                    fcg_commit(st[sys], s, prev, f, hd.iter0 + idx, active);
                else if (f.off)
                    st[sys].precOff = 1;
            }
        }
        __syncthreads();
        if (pause) return;
        betaD = bc[0];
    }
    if (blockIdx.x == 0 && blockIdx.y % FL == 0 && threadIdx.x == 0) st[sys].ab[idx & 1].y = rz;
    const float beta = (float)betaD;
#pragma unroll
    for (int u = 0; u < M0; ++u) {
        const int i = threadIdx.x + u * NT;
        if (i < N) {
            d[u] = (float)A.d0 + (float)A.g * d[u];
            p[u] = axpy<float>(q[u], beta, p[u]);
            P.set(i, p[u]);
            if (place[u] & 2) store_sp<float>(pnew, V, g[u], p[u]);
        }
    }
    __syncthreads();
    double mu = 0.0;
#pragma unroll
    for (int u = 0; u < M0; ++u)
        if (place[u] & 1) {
            const int i = threadIdx.x + u * NT;
            q[u] = pl_dirac<float, false, WR1>((float)A.r, P, i, W, place[u] & 4 ? -1.f : 1.f,
                                               place[u] & 8 ? -1.f : 1.f, d[u], p[u]);
            Q.set(i, q[u]);
            if (place[u] & 2) mu += sq(q[u]);
        }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < M0; ++u)
        if (place[u] & 2)
            store_sp<float>(Ap, V, g[u],
                            pl_dirac<float, true, WR1>((float)A.r, Q, threadIdx.x + u * NT, W,
                                                       place[u] & 4 ? -1.f : 1.f, place[u] & 8 ? -1.f : 1.f, d[u],
                                                       q[u]));
    const double v = block_sum3<NT>(mu, 0.0, 0.0, red);
    if (threadIdx.x == 0) part[(size_t)blockIdx.y * gridDim.x + blockIdx.x] = v;
}

// after the last of a chunk's n iterations: its state, for the reliable update
__global__ void __launch_bounds__(kPfNT)
k_fcg_close(const double2 *__restrict__ cnnPart, int nb, int n, CgState *__restrict__ st, int *__restrict__ active) {
    __shared__ double red[3 * kPfNT / kWave];
    CgState &S = st[blockIdx.x];
    const PfHead hd = pf_head(S);
    const Pf3 s = sum_pf_partials<kPfNT>(cnnPart + 2 * (size_t)blockIdx.x * nb, nb, red);
    if (hd.done || threadIdx.x) return;
    const double2 prev = S.ab[(n - 1) & 1];
    fcg_commit(S, s, prev, fcg_decide(s, prev, hd.iter0 + n, hd), hd.iter0 + n, active);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// Tiles and their block sizes.  Lattices that fill the chip want few waves per block, each with two
// to four entries, so that several blocks share a compute unit and one loads while another works:
// at 1024 x 1024 in FP64 8x32 takes 31.8 us with 256 threads and 36.1 with 448 (one entry each),
// 16x32 32.3 and 40.9 with 384.  A persistent grid that prefetches the next tile was no faster
// (32.4 at best).
struct PlTile {
    int TT, TX, NT;
};
constexpr PlTile kPlTiles[] = {{4, 16, 192}, {8, 32, 256}, {16, 16, 256}, {16, 32, 256}, {32, 32, 448}, {8, 64, 256},
                               {16, 64, 704}};
constexpr int kNumPl = sizeof(kPlTiles) / sizeof(kPlTiles[0]);
// FP64 only: tiles of k_pl_rc, numbered after those.  The entries per thread (two) matter more than
// the tile: 16x32 with 960 threads takes 43.9 us at 1024 x 1024, with 256 35.1.
constexpr PlTile kRcTiles[] = {{16, 32, 512}, {32, 32, 832}, {16, 64, 896}};
constexpr int kNumRc = sizeof(kRcTiles) / sizeof(kRcTiles[0]);
static PlTile pl_tile(int i) { return i < kNumPl ? kPlTiles[i] : kRcTiles[i - kNumPl]; }

// a tile need not divide the lattice, but its halo may wrap around only once
static bool pl_fits(const Ctx &c, int i) {
    const PlTile t = pl_tile(i);
    const int halo = i < kNumPl ? 2 : 4;
    auto ok = [&](int n, int T) { return n >= halo && (n % T == 0 || n > T + halo - 2); };
    return ok(c.p.Nt, t.TT) && ok(c.p.Nx, t.TX);
}
static int pl_blocks(const Ctx &c, PlTile t) {
    return ((c.p.Nt + t.TT - 1) / t.TT) * ((c.p.Nx + t.TX - 1) / t.TX);
}

template <typename R>
struct PlPtrs {
    using V2 = typename Vec2<R>::T;
    const R *phi;
    const V2 *r, *Ap_in, *pold;
    V2 *pnew, *Ap, *x;
};

static PlArgs pl_args(const Ctx &c, int TT, int TX) {
    PlArgs A;
    A.Nt = c.p.Nt;
    A.Nx = c.p.Nx;
    A.V = c.V;
    A.nNoise = c.nNoise;
    A.r = c.p.r;
    A.d0 = 2.0 * c.p.r + c.p.M;
    A.g = c.p.g;
    A.tilesX = (c.p.Nx + TX - 1) / TX;
    A.tilesPerSys = pl_blocks(c, {TT, TX, 0});
    A.xcdRemap = A.tilesPerSys % 8 == 0 ? 1 : 0;
    return A;
}

// launch idx of a chunk; form 0: launch 0 of a phase (r read), 1: odd launches, 2: even ones;
// returns the block partials per system
template <typename R, int TT, int TX, int NT>
static int launch_pl_tt(const Ctx &c, int nsys, bool dag1, int idx, int form, int finMode, const PlPtrs<R> &b) {
    PlArgs A = pl_args(c, TT, TX);
    auto go = [&](auto dagTag, auto wrTag) {
        constexpr bool D = decltype(dagTag)::value, W1 = decltype(wrTag)::value;
        using K = decltype(&k_pl_pf<R, TT, TX, NT, D, W1, 0, 1>);
        const K ks[3] = {&k_pl_pf<R, TT, TX, NT, D, W1, 0, 1>, &k_pl_pf<R, TT, TX, NT, D, W1, 2, 2>,
                         &k_pl_pf<R, TT, TX, NT, D, W1, 0, 2>};
        hipLaunchKernelGGL(ks[form], dim3(A.tilesPerSys, nsys), dim3(NT), 0, c.stream, A, b.phi, c.cg_d, b.r, b.Ap_in,
                           b.pold, b.pnew, b.Ap, b.x, c.pfSlot[idx & 1], finMode, idx,
                           (const double2 *)c.pfSlot[~idx & 1], c.active);
    };
    const bool w1 = c.p.r == 1.0;
    if (dag1)
        w1 ? go(std::true_type(), std::true_type()) : go(std::true_type(), std::false_type());
    else
        w1 ? go(std::false_type(), std::true_type()) : go(std::false_type(), std::false_type());
    return A.tilesPerSys;
}

// k_pl_rc for the launches after a phase's first
template <int TT, int TX, int NT>
static int launch_rc_tt(const Ctx &c, int nsys, bool dag1, int idx, int form, int finMode, const PlPtrs<double> &b) {
    if (form == 0) return launch_pl_tt<double, TT, TX, NT>(c, nsys, dag1, idx, form, finMode, b);
    PlArgs A = pl_args(c, TT, TX);
    auto go = [&](auto dagTag, auto wrTag) {
        constexpr bool D = decltype(dagTag)::value, W1 = decltype(wrTag)::value;
        auto *k = form == 1 ? &k_pl_rc<double, TT, TX, NT, D, W1, 2> : &k_pl_rc<double, TT, TX, NT, D, W1, 0>;
        hipLaunchKernelGGL(k, dim3(A.tilesPerSys, nsys), dim3(NT), 0, c.stream, A, b.phi, c.cg_d, b.r, b.pold, b.pnew,
                           b.x, c.pfSlot[idx & 1], finMode, idx, (const double2 *)c.pfSlot[~idx & 1], c.active);
    };
    const bool w1 = c.p.r == 1.0;
    if (dag1)
        w1 ? go(std::true_type(), std::true_type()) : go(std::true_type(), std::false_type());
    else
        w1 ? go(std::false_type(), std::true_type()) : go(std::false_type(), std::false_type());
    return A.tilesPerSys;
}

static int launch_rc(const Ctx &c, int ti, int nsys, bool dag1, int idx, int form, int finMode,
                     const PlPtrs<double> &b) {
    switch (ti - kNumPl) {
    case 0: return launch_rc_tt<16, 32, 512>(c, nsys, dag1, idx, form, finMode, b);
    case 1: return launch_rc_tt<32, 32, 832>(c, nsys, dag1, idx, form, finMode, b);
    default: return launch_rc_tt<16, 64, 896>(c, nsys, dag1, idx, form, finMode, b);
    }
}

template <typename R>
static int launch_pl_any(Ctx &c, int ti, int nsys, bool dag1, int idx, int form, int finMode, const PlPtrs<R> &b) {
    const PlTile t = pl_tile(ti);
    prof_before(c, PK_NORMAL_OP, (double)nsys * c.V * ((idx & 1 ? 7 : 5) * 4 - (ti < kNumPl ? 0 : 8) + 1) * sizeof(R));
    int nb = 0;
    if (ti >= kNumPl) {
        if constexpr (std::is_same<R, double>::value) nb = launch_rc(c, ti, nsys, dag1, idx, form, finMode, b);
        prof_after(c, PK_NORMAL_OP);
        return nb;
    }
    switch (t.TT * 1000 + t.TX) {
    case 4016: nb = launch_pl_tt<R, 4, 16, 192>(c, nsys, dag1, idx, form, finMode, b); break;
    case 8032: nb = launch_pl_tt<R, 8, 32, 256>(c, nsys, dag1, idx, form, finMode, b); break;
    case 16016: nb = launch_pl_tt<R, 16, 16, 256>(c, nsys, dag1, idx, form, finMode, b); break;
    case 16032: nb = launch_pl_tt<R, 16, 32, 256>(c, nsys, dag1, idx, form, finMode, b); break;
    case 32032: nb = launch_pl_tt<R, 32, 32, 448>(c, nsys, dag1, idx, form, finMode, b); break;
    case 8064: nb = launch_pl_tt<R, 8, 64, 256>(c, nsys, dag1, idx, form, finMode, b); break;
    default: nb = launch_pl_tt<R, 16, 64, 704>(c, nsys, dag1, idx, form, finMode, b); break;
    }
    prof_after(c, PK_NORMAL_OP);
    return nb;
}

// FP32 launch idx of a chunk (buffers as in the even-odd iteration's launch_eo_pf, on the full
// lattice)
static int launch_pl(Ctx &c, int ti, int nsys, bool dag1, int idx, int finMode) {
    const int par = idx & 1;
    PlPtrs<float> b;
    b.phi = c.phis;
    b.r = idx == 0 ? c.rs : pf_dir(c, idx - 2);
    b.Ap_in = par ? c.pfA1 : c.Aps;
    b.pold = pf_dir(c, idx - 1);
    b.pnew = pf_dir(c, idx);
    b.Ap = par ? c.Aps : c.pfA1;
    b.x = c.xs;
    return launch_pl_any<float>(c, ti, nsys, dag1, idx, idx == 0 ? 0 : par ? 1 : 2, finMode, b);
}

// FP64 direction p_k of a phase: p[0] (p_{-1}, multiplied by 0), p[1], and r, which nothing reads
// after launch 0
static double2 *p64_dir(const Ctx &c, int k) {
    double2 *const rot[3] = {c.pv[0], c.pv[1], c.r};
    return rot[(k + 1) % 3];
}
// FP64 launch idx of a chunk (first: the phase's first), A p alternating between t and Ap
static int launch_p64(Ctx &c, int ti, int nsys, const double *phi, bool dag1, int idx, bool first, int finMode) {
    const int par = idx & 1;
    PlPtrs<double> b;
    b.phi = phi;
    b.r = first && idx == 0 ? c.r : p64_dir(c, idx + 1);   // p_{idx-2}
    b.Ap_in = par ? c.t : c.Ap;
    b.pold = p64_dir(c, idx + 2);
    b.pnew = p64_dir(c, idx);
    b.Ap = par ? c.Ap : c.t;
    b.x = c.x;
    return launch_pl_any<double>(c, ti, nsys, dag1, idx, first && idx == 0 ? 0 : par ? 1 : 2, finMode, b);
}
// the partial slots, and for mixed precision the buffers beyond the mixed solver's: second Ap,
// third direction
static int pl_alloc(Ctx &c, bool mixed) {
    size_t nb = 0;
    for (int i = 0; i < kNumPl + kNumRc; ++i)
        if (pl_fits(c, i)) nb = std::max(nb, (size_t)pl_blocks(c, pl_tile(i)));
    if (!nb || c.V >= (1 << 27)) return YCN_OK;   // 32-bit byte offsets into a system's two planes
    const size_t n = (size_t)c.nSys * kPacked * c.V;
    if (mixed)
        for (float2 **b : {&c.pfA1, &c.pfP2}) {
            YCN_HIP(hipMalloc(b, sizeof(float2) * n));
            YCN_HIP(hipMemset(*b, 0, sizeof(float2) * n));
        }
    for (double2 *&slot : c.pfSlot) {
        YCN_HIP(hipMalloc(&slot, sizeof(double2) * c.nSys * nb * 2));
        YCN_HIP(hipMemset(slot, 0, sizeof(double2) * c.nSys * nb * 2));
    }
    return YCN_OK;
}

// (neither has an update kernel of its own to time)
bool pl_available(const Ctx &c) { return c.tilePl >= 0 && c.profTarget != PK_CG_UPDATE; }
bool p64_available(const Ctx &c) { return c.tileP64 >= 0 && c.profTarget != PK_CG_UPDATE; }

// The pipelined iteration of the context's precision: times every tile that fits, with either
// finalize, and keeps the fastest pair.
int pl_autotune(Ctx &c) {
    c.tilePl = c.tileP64 = -1;
    if (c.p.evenOdd || c.p.precond != YCN_PRECOND_NONE || onchip_plain(c)) return YCN_OK;
    const bool mixed = c.p.cgPrecision == YCN_CG_MIXED;
    if (std::getenv(mixed ? "YCN_TILE32" : "YCN_TILE")) return YCN_OK;   // a forced tile of the unpipelined iteration
    const int rc = pl_alloc(c, mixed);
    if (rc || !c.pfSlot[1]) return rc;
    std::vector<double> us;
    const int memoKey = mixed ? 2 : 3, n = mixed ? kNumPl : kNumPl + kNumRc;
    const bool memo = tune_lookup(memoKey, c, us) && us.size() == 2 * (size_t)n;
    if (!memo) {
        us.assign(2 * n, 1e30);
        hipEvent_t e0, e1;
        YCN_HIP(hipEventCreate(&e0));
        YCN_HIP(hipEventCreate(&e1));
        YCN_HIP(hipMemsetAsync(c.cg_d, 0, sizeof(CgState) * c.nSys, c.stream));
        const int reps = c.V >= (1 << 16) ? 10 : 4;
        for (int i = 0; i < n; ++i) {
            if (!pl_fits(c, i)) continue;
            for (int m = 0; m < 2; ++m) {
                auto launch = [&](int k) {
                    const int nb = mixed ? launch_pl(c, i, c.nSys, false, k, m ? 2 : 0)
                                         : launch_p64(c, i, c.nSys, c.phi[c.cur], false, k, true, m ? 2 : 0);
                    if (!m && mixed) launch_fin_pf(c, c.nSys, nb, 0, c.pfSlot[k & 1]);
                    if (!m && !mixed) launch_fin_p64(c, c.nSys, nb, 1, c.pfSlot[k & 1], 0);
                };
                launch(0);
                launch(1);
                (void)hipEventRecord(e0, c.stream);
                for (int k = 0; k < reps; ++k) launch(2 + k);
                (void)hipEventRecord(e1, c.stream);
                (void)hipEventSynchronize(e1);
                float ms = 0;
                (void)hipEventElapsedTime(&ms, e0, e1);
                us[2 * i + m] = 1e3 * ms / reps;
            }
        }
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        YCN_HIP(hipGetLastError());
        YCN_HIP(hipMemsetAsync(c.cg_d, 0, sizeof(CgState) * c.nSys, c.stream));
        YCN_HIP(hipStreamSynchronize(c.stream));
        tune_store(memoKey, c, us);
    }
    const char *force = std::getenv("YCN_TILE_PL");   // forces a tile of the table (tests cover every one)
    const int f = force ? std::atoi(force) : -1;
    char line[96];
    double best = 1e30;
    int &tile = mixed ? c.tilePl : c.tileP64;
    c.tuneReport += mixed ? " | fp32 pipelined tiles (us/iteration, separate | prologue finalize):"
                          : " | fp64 pipelined tiles (us/iteration, separate | prologue finalize):";
    for (int i = 0; i < n; ++i) {
        if (!pl_fits(c, i)) continue;
        std::snprintf(line, sizeof line, " %dx%d%s %.1f|%.1f;", pl_tile(i).TT, pl_tile(i).TX, i < kNumPl ? "" : "r",
                      us[2 * i], us[2 * i + 1]);
        c.tuneReport += line;
        for (int m = 0; m < 2; ++m)
            if ((f < 0 || f == i) && us[2 * i + m] < best) {
                best = us[2 * i + m];
                tile = i;
                c.eoFinFused = m == 1;
            }
    }
    if (const char *fin = std::getenv("YCN_PL_FIN")) c.eoFinFused = std::strcmp(fin, "fused") == 0;
    if (tile >= 0) {
        const PlTile t = pl_tile(tile);
        tune_report_choice(c, mixed ? "fp32" : "fp64", t.TT, t.TX, tile < kNumPl ? "" : "r");
    }
    return YCN_OK;
}

// n FP32 iterations of a chunk on the systems, from the context's residual and kept direction
int pl_iterations(Ctx &c, int nsys, int mtype, int n) {
    const bool dag1 = mtype != YCN_DAGGER;
    const int rc = run_chunk(c, nullptr, nsys, mtype, n, 5, kPacked, c.tilePl, [&](int i) {
        const int nb = launch_pl(c, c.tilePl, nsys, dag1, i, c.eoFinFused ? 1 : 0);
        if (!c.eoFinFused) launch_fin_pf(c, nsys, nb, 1, c.pfSlot[i & 1]);
    });
    if (rc) return rc;
    c.eoPfBlocks = pl_blocks(c, pl_tile(c.tilePl));
    return YCN_OK;
}

// One captured chunk of FP64 iterations (first: of a phase, from the residual in r); returns the
// launches in *n.  A phase is what runs until every system has stopped; p64_close ends it.
int p64_iterations(Ctx &c, const double *phi, int nsys, int mtype, bool first, int *n) {
    *n = kP64Launches;
    const bool dag1 = mtype != YCN_DAGGER, fused = c.eoFinFused;
    return run_chunk(c, phi, nsys, mtype, kP64Launches, first ? 6 : 7, kPacked, c.tileP64, [&](int i) {
        const int nb = launch_p64(c, c.tileP64, nsys, phi, dag1, i, first, fused ? 1 : 0);
        if (!fused || i == kP64Launches - 1)
            launch_fin_p64(c, nsys, nb, fused ? kP64Launches : 1, c.pfSlot[i & 1], 1);
    });
}
void p64_close(Ctx &c, int nsys) {
    hipLaunchKernelGGL(k_p64_close<false>, dim3((c.V + kPfNT - 1) / kPfNT, nsys), dim3(kPfNT), 0, c.stream, c.V,
                       (const CgState *)c.cg_d, c.x, c.pv[0], (const double2 *)c.pv[1], c.r, (const double2 *)nullptr,
                       (const double2 *)nullptr);
}

// iteration idx of a chunk of the flexible solver (see k_fcg_op): r and the directions alternate
// between two buffers, both ways starting from the first
int fcg_iteration(Ctx &c, SpinorForm form, int nsys, int idx) {
    PlArgs A = pl_args(c, 16, 16);
    const int par = idx & 1, tiles = A.tilesPerSys;
    double *const opPart = reinterpret_cast<double *>(c.partials + (size_t)2 * nsys * tiles);
    const int fl = form == kPacked ? 1 : 2;
    prof_before(c, PK_NORMAL_OP, (double)nsys * c.V * (4 * 16 * fl + 4));
    auto *k = form == kPacked ? (A.r == 1.0 ? &k_fcg_op<true, 1> : &k_fcg_op<false, 1>)
                              : (A.r == 1.0 ? &k_fcg_op<true, 2> : &k_fcg_op<false, 2>);
    hipLaunchKernelGGL(k, dim3(tiles, fl * nsys), dim3(kFcgNT), 0, c.stream, A, (const float *)c.phis, c.cg_d,
                       (const float2 *)c.zs, (const float2 *)c.ps[par], c.ps[par ^ 1], c.Aps, opPart, idx,
                       (const double2 *)c.partials, tiles, c.active);
    prof_after(c, PK_NORMAL_OP);
    FcgUpdate u;
    u.rnew = par ? c.rs : c.pfA1;
    u.p = c.ps[par ^ 1];
    u.xs = c.xs;
    u.opPart = opPart;
    u.nbOp = fl * tiles;
    u.idx = idx;
    return cnn_update_apply(c, form, nsys, par ? c.pfA1 : c.rs, u);
}
void fcg_close(Ctx &c, int nsys, int n) {
    hipLaunchKernelGGL(k_fcg_close, dim3(nsys), dim3(kPfNT), 0, c.stream, (const double2 *)c.partials,
                       (c.p.Nt / 16) * (c.p.Nx / 16), n, c.cg_d, c.active);
}

}  // namespace ycn
