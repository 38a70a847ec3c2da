// plain.hip -- the pipelined FP32 iteration of the plain mixed-precision solver on D^dag D or
// D D^dag (packed real spinors): one launch per CG iteration.
//
// The iteration is the even-odd one's (k_eo_normal_fused in evenodd.hip): CG with the residual
// norm recurrence of D'Azevedo, Eijkhout and Romine (LAPACK Working Note 56, 1993), so that one
// reduction per iteration suffices and the x and r updates move into the next application of
// the operator; r rebuilt from the directions after launch 0 of a chunk, x_s updated by every
// other launch for both; the finalize in the next launch's prologue or a launch of its own.
// Per site and launch it reads p_{k-2} (or r), Ap, p and phi and writes p and Ap, and every other
// launch updates x_s: 84 and 116 B, against 4 x 16 + 4 and 6 x 16 B in four launches (operator,
// alpha, update, beta) before.
//
// What bounds it: at 512 x 512 the vectors stay in the caches and a launch is latency, its chain
// of partial sums, loads, two stencil stages and a reduction.
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "cg_fused.hpp"
#include "pipelined.hpp"

namespace ycn {

struct PlArgs {
    int Nt, Nx, V, nNoise;
    float hp, hm, hr, d0, g;
    int tilesX, tilesPerSys, xcdRemap;
};

// v times d minus the hop of D (DAG = false) or D^dag at array entry i of N (rows of W)
template <bool DAG, bool WR1>
__device__ __forceinline__ float4 pl_dirac(const PlArgs &A, const float4 *N, int i, int W, float sf, float sb, float d,
                                           float4 v) {
    const float2 *const N2 = reinterpret_cast<const float2 *>(N);
    const float sTb = DAG ? sf : sb, sTf = DAG ? sb : sf;
    const int iTb = DAG ? i + W : i - W, iTf = DAG ? i - W : i + W;
    const float4 xf = DAG ? N[i - 1] : N[i + 1], xb = DAG ? N[i + 1] : N[i - 1];
    const float2 tb0 = N2[2 * iTb], tf1 = N2[2 * iTf + 1];
    float4 o;
    if constexpr (WR1) {
        o.x = sTb * tb0.x + 0.5f * ((xf.x + xb.x) + (xb.z - xf.z));
        o.y = sTb * tb0.y + 0.5f * ((xf.y + xb.y) + (xb.w - xf.w));
        o.z = sTf * tf1.x + 0.5f * ((xf.z + xb.z) + (xb.x - xf.x));
        o.w = sTf * tf1.y + 0.5f * ((xf.w + xb.w) + (xb.y - xf.y));
    } else {
        const float2 tb1 = N2[2 * iTb + 1], tf0 = N2[2 * iTf];
        const float ap = A.hp * sTb, am = A.hm * sTf, bm = A.hm * sTb, bp = A.hp * sTf;
        o.x = ap * tb0.x + am * tf0.x + A.hr * (xf.x + xb.x) + 0.5f * (xb.z - xf.z);
        o.y = ap * tb0.y + am * tf0.y + A.hr * (xf.y + xb.y) + 0.5f * (xb.w - xf.w);
        o.z = bm * tb1.x + bp * tf1.x + A.hr * (xf.z + xb.z) + 0.5f * (xb.x - xf.x);
        o.w = bm * tb1.y + bp * tf1.y + A.hr * (xf.w + xb.w) + 0.5f * (xb.y - xf.y);
    }
    return make_float4(d * v.x - o.x, d * v.y - o.y, d * v.z - o.z, d * v.w - o.w);
}
__device__ __forceinline__ float sq4(float4 v) { return (v.x * v.x + v.y * v.y) + (v.z * v.z + v.w * v.w); }
__device__ __forceinline__ float4 axpy4(float4 u, float s, float4 v) {
    return make_float4(u.x + s * v.x, u.y + s * v.y, u.z + s * v.z, u.w + s * v.w);
}

// One launch of the iteration; XM, RM, idx and finMode as in k_eo_normal_fused.  A block owns a
// TT x TX tile; a thread keeps the same M0 entries of the tile with its 2-site halo through all
// stages, so that an entry's own values stay in registers.
template <int TT, int TX, int NT, bool DAG1, bool WR1, int XM, int RM>
__global__ void __launch_bounds__(NT)
k_pl_pf(PlArgs A, const float *__restrict__ phi, CgState *st, const float2 *__restrict__ r,
        const float2 *__restrict__ Ap_in, const float2 *__restrict__ pold, float2 *__restrict__ pnew,
        float2 *__restrict__ Ap, float2 *__restrict__ xs, double2 *__restrict__ part, int finMode, int idx,
        const double2 *__restrict__ prevPart, int *active) {
    constexpr int H = TT + 4, W = TX + 4, N = H * W, M0 = (N + NT - 1) / NT;
    __shared__ float4 P[N], Q[N];
    __shared__ double2 red[NT / kWave], red2[NT / kWave];
    __shared__ double bc[3];
    __shared__ int pause;
    const int sys = blockIdx.y;
    if (st[sys].done) return;
    const unsigned V = (unsigned)A.V;
    const size_t off = (size_t)sys * 2 * V;
    r += off;
    Ap_in += off;
    pold += off;
    pnew += off;
    Ap += off;
    xs += off;
    const float *ph = phi + (size_t)(sys / A.nNoise) * V;
    int tile = blockIdx.x;   // contiguous bands of tiles per XCD
    if (A.xcdRemap) tile = (tile % 8) * (A.tilesPerSys / 8) + tile / 8;
    const int ty = tile / A.tilesX, t0 = ty * TT, x0 = (tile - ty * A.tilesX) * TX;

    // an entry's place: 1 = within the 1-site halo, 2 = the tile's own; 4, 8: the hops across
    // the time boundary, forward and backward
    float4 a[M0], p[M0], q[M0], xv[M0];
    float d[M0];
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
            const bool in2 = row >= 2 && row < H - 2 && col >= 2 && col < W - 2;
            at_[u] = (in1 ? 1 : 0) | (in2 ? 2 : 0) | (gt == A.Nt - 1 ? 4 : 0) | (gt == 0 ? 8 : 0);
            const float2 r0 = at(r, gs[u]), r1 = at(r, V + gs[u]), p0 = at(pold, gs[u]), p1 = at(pold, V + gs[u]),
                         q0 = at(Ap_in, gs[u]), q1 = at(Ap_in, V + gs[u]);
            a[u] = make_float4(r0.x, r0.y, r1.x, r1.y);
            p[u] = make_float4(p0.x, p0.y, p1.x, p1.y);
            q[u] = make_float4(q0.x, q0.y, q1.x, q1.y);
            if (XM != 0 && in2) {
                const float2 x0_ = at(xs, gs[u]), x1_ = at(xs, V + gs[u]);
                xv[u] = make_float4(x0_.x, x0_.y, x1_.x, x1_.y);
            }
            d[u] = at(ph, gs[u]);
        }
    }
    const double2 prev = RM == 2 ? st[sys].ab[(idx - 1) & 1] : make_double2(0.0, 0.0);
    double alphaD, betaD;
    if (!pf_prologue<NT>(st, sys, idx, finMode, prevPart, part, active, red, red2, bc, &pause, alphaD, betaD)) return;
    if (blockIdx.x == 0 && threadIdx.x == 0) st[sys].ab[idx & 1] = make_double2(alphaD, betaD);
    const float alpha = (float)alphaD, beta = (float)betaD, alphaPrev = (float)prev.x, betaPrev = (float)prev.y;

    double rho = 0.0, mu = 0.0, nu = 0.0;
#pragma unroll
    for (int u = 0; u < M0; ++u) {
        const int i = threadIdx.x + u * NT;
        if (i < N) {
            d[u] = A.d0 + A.g * d[u];
            const float4 p2 = a[u];
            if (RM == 2) a[u] = axpy4(p[u], -betaPrev, a[u]);
            a[u] = axpy4(a[u], -alpha, q[u]);
            if (at_[u] & 2) {
                rho += (double)sq4(a[u]);
                if (XM == 2) {
                    xv[u] = axpy4(axpy4(xv[u], alphaPrev, p2), alpha, p[u]);
                    at(xs, gs[u]) = make_float2(xv[u].x, xv[u].y);
                    at(xs, V + gs[u]) = make_float2(xv[u].z, xv[u].w);
                }
            }
            p[u] = axpy4(a[u], beta, p[u]);
            P[i] = p[u];
            if (at_[u] & 2) {
                at(pnew, gs[u]) = make_float2(p[u].x, p[u].y);
                at(pnew, V + gs[u]) = make_float2(p[u].z, p[u].w);
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < M0; ++u)
        if (at_[u] & 1) {
            const int i = threadIdx.x + u * NT;
            q[u] = pl_dirac<DAG1, WR1>(A, P, i, W, at_[u] & 4 ? -1.f : 1.f, at_[u] & 8 ? -1.f : 1.f, d[u], p[u]);
            Q[i] = q[u];
            if (at_[u] & 2) mu += (double)sq4(q[u]);
        }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < M0; ++u)
        if (at_[u] & 2) {
            const int i = threadIdx.x + u * NT;
            const float4 o = pl_dirac<!DAG1, WR1>(A, Q, i, W, at_[u] & 4 ? -1.f : 1.f, at_[u] & 8 ? -1.f : 1.f, d[u],
                                                  q[u]);
            at(Ap, gs[u]) = make_float2(o.x, o.y);
            at(Ap, V + gs[u]) = make_float2(o.z, o.w);
            nu += (double)sq4(o);
        }
    const size_t pidx = (size_t)sys * gridDim.x + blockIdx.x;
    const double2 t1 = block_sum2<NT>(make_double2(mu, nu), red);
    const double2 t2 = block_sum2<NT>(make_double2(rho, 0.0), red2);
    if (threadIdx.x == 0) {
        part[2 * pidx] = t1;
        part[2 * pidx + 1] = t2;
    }
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// Tiles and the block sizes that their entries (with the halo) divide into with few idle threads.
struct PlTile {
    int TT, TX, NT;
};
constexpr PlTile kPlTiles[] = {{4, 16, 192}, {8, 32, 448}, {16, 16, 448}, {16, 32, 384}, {32, 32, 448}, {8, 64, 448},
                               {16, 64, 704}};
constexpr int kNumPl = sizeof(kPlTiles) / sizeof(kPlTiles[0]);

static bool pl_fits(const Ctx &c, PlTile t) { return c.p.Nt % t.TT == 0 && c.p.Nx % t.TX == 0; }

// launch idx of a chunk (buffers as in the even-odd iteration's launch_eo_pf, on the full
// lattice); returns the block partials per system
template <int TT, int TX, int NT>
static int launch_pl_tt(const Ctx &c, int nsys, bool dag1, int idx, int finMode) {
    PlArgs A;
    A.Nt = c.p.Nt;
    A.Nx = c.p.Nx;
    A.V = c.V;
    A.nNoise = c.nNoise;
    A.hp = (float)(0.5 * (c.p.r + 1.0));
    A.hm = (float)(0.5 * (c.p.r - 1.0));
    A.hr = (float)(0.5 * c.p.r);
    A.d0 = (float)(2.0 * c.p.r + c.p.M);
    A.g = (float)c.p.g;
    A.tilesX = c.p.Nx / TX;
    A.tilesPerSys = (c.p.Nt / TT) * A.tilesX;
    A.xcdRemap = A.tilesPerSys % 8 == 0 ? 1 : 0;
    const int par = idx & 1, form = idx == 0 ? 0 : par ? 1 : 2;
    const float2 *r = idx == 0 ? c.rs : pf_dir(c, idx - 2);
    double2 *part = finMode ? c.pfSlot[par] : c.partials;
    auto go = [&](auto dagTag, auto wrTag) {
        constexpr bool D = decltype(dagTag)::value, W1 = decltype(wrTag)::value;
        using K = decltype(&k_pl_pf<TT, TX, NT, D, W1, 0, 1>);
        const K ks[3] = {&k_pl_pf<TT, TX, NT, D, W1, 0, 1>, &k_pl_pf<TT, TX, NT, D, W1, 2, 2>,
                         &k_pl_pf<TT, TX, NT, D, W1, 0, 2>};
        hipLaunchKernelGGL(ks[form], dim3(A.tilesPerSys, nsys), dim3(NT), 0, c.stream, A, (const float *)c.phis, c.cg_d,
                           r, (const float2 *)(par ? c.pfA1 : c.Aps), (const float2 *)pf_dir(c, idx - 1),
                           pf_dir(c, idx), par ? c.Aps : c.pfA1, c.xs, part, finMode, idx,
                           (const double2 *)c.pfSlot[par ^ 1], c.active);
    };
    const bool w1 = c.p.r == 1.0;
    if (dag1)
        w1 ? go(std::true_type(), std::true_type()) : go(std::true_type(), std::false_type());
    else
        w1 ? go(std::false_type(), std::true_type()) : go(std::false_type(), std::false_type());
    return A.tilesPerSys;
}

static int launch_pl(Ctx &c, int ti, int nsys, bool dag1, int idx, int finMode) {
    const PlTile t = kPlTiles[ti];
    prof_before(c, PK_NORMAL_OP, (double)nsys * c.V * ((idx & 1 ? 7 : 5) * 16 + 4));
    int nb = 0;
    switch (t.TT * 1000 + t.TX) {
    case 4016: nb = launch_pl_tt<4, 16, 192>(c, nsys, dag1, idx, finMode); break;
    case 8032: nb = launch_pl_tt<8, 32, 448>(c, nsys, dag1, idx, finMode); break;
    case 16016: nb = launch_pl_tt<16, 16, 448>(c, nsys, dag1, idx, finMode); break;
    case 16032: nb = launch_pl_tt<16, 32, 384>(c, nsys, dag1, idx, finMode); break;
    case 32032: nb = launch_pl_tt<32, 32, 448>(c, nsys, dag1, idx, finMode); break;
    case 8064: nb = launch_pl_tt<8, 64, 448>(c, nsys, dag1, idx, finMode); break;
    default: nb = launch_pl_tt<16, 64, 704>(c, nsys, dag1, idx, finMode); break;
    }
    prof_after(c, PK_NORMAL_OP);
    return nb;
}

// the buffers beyond the mixed solver's: second Ap, third direction, the partial slots of
// prologue-finalized launches (64-site tiles at the smallest)
int pl_alloc(Ctx &c) {
    bool any = false;
    for (const PlTile &t : kPlTiles) any = any || pl_fits(c, t);
    if (!any || c.V >= (1 << 27)) return YCN_OK;   // 32-bit byte offsets into a system's two planes
    const size_t n = (size_t)c.nSys * kPacked * c.V;
    for (float2 **b : {&c.pfA1, &c.pfP2}) {
        YCN_HIP(hipMalloc(b, sizeof(float2) * n));
        YCN_HIP(hipMemset(*b, 0, sizeof(float2) * n));
    }
    return eo_pf_alloc(c);
}

bool pl_available(const Ctx &c) { return c.tilePl >= 0; }

// times every tile that fits, with either finalize, and keeps the fastest pair
int pl_autotune(Ctx &c) {
    c.tilePl = -1;
    if (c.p.evenOdd || !c.rs || !c.pfA1 || !c.pfP2 || !c.pfSlot[1]) return YCN_OK;
    std::vector<double> us;
    const bool memo = tune_lookup(2, c, us) && us.size() == 2 * (size_t)kNumPl;
    if (!memo) {
        us.assign(2 * kNumPl, 1e30);
        hipEvent_t e0, e1;
        YCN_HIP(hipEventCreate(&e0));
        YCN_HIP(hipEventCreate(&e1));
        YCN_HIP(hipMemsetAsync(c.cg_d, 0, sizeof(CgState) * c.nSys, c.stream));
        const int reps = c.V >= (1 << 16) ? 10 : 4;
        for (int i = 0; i < kNumPl; ++i) {
            if (!pl_fits(c, kPlTiles[i])) continue;
            for (int m = 0; m < 2; ++m) {
                auto launch = [&](int k) {
                    const int nb = launch_pl(c, i, c.nSys, false, k, m ? 2 : 0);
                    if (!m) launch_fin_pf(c, c.nSys, nb, 0);
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
        tune_store(2, c, us);
    }
    const char *force = std::getenv("YCN_TILE_PL");   // forces a tile of the table (tests cover every one)
    const int f = force ? std::atoi(force) : -1;
    char line[96];
    double best = 1e30;
    c.tuneReport += " | fp32 pipelined tiles (us/iteration, separate | prologue finalize):";
    for (int i = 0; i < kNumPl; ++i) {
        if (!pl_fits(c, kPlTiles[i])) continue;
        std::snprintf(line, sizeof line, " %dx%d %.1f|%.1f;", kPlTiles[i].TT, kPlTiles[i].TX, us[2 * i], us[2 * i + 1]);
        c.tuneReport += line;
        for (int m = 0; m < 2; ++m)
            if ((f < 0 || f == i) && us[2 * i + m] < best) {
                best = us[2 * i + m];
                c.tilePl = i;
                c.eoFinFused = m == 1;
            }
    }
    if (const char *fin = std::getenv("YCN_PL_FIN")) c.eoFinFused = std::strcmp(fin, "fused") == 0;
    return YCN_OK;
}

// n iterations of a chunk on the systems, from the context's residual and kept direction
int pl_iterations(Ctx &c, int nsys, int mtype, int n) {
    const bool dag1 = mtype != YCN_DAGGER;
    const int rc = run_chunk(c, nullptr, nsys, mtype, n, 5, kPacked, c.tilePl, [&](int i) {
        const int nb = launch_pl(c, c.tilePl, nsys, dag1, i, c.eoFinFused ? 1 : 0);
        c.eoPfBlocks = nb;
        if (!c.eoFinFused) launch_fin_pf(c, nsys, nb, 1);
    });
    if (rc) return rc;
    c.eoPfBlocks = (c.p.Nt / kPlTiles[c.tilePl].TT) * (c.p.Nx / kPlTiles[c.tilePl].TX);
    if (c.eoFinFused) launch_fin_pf_chunk(c, nsys, n);
    return YCN_OK;
}

}  // namespace ycn
