// evenodd.hip -- even-odd preconditioned fermion force on gfx950.
//
// The drift only needs chi = (D^dag)^-1 eta (chi = D y with D^dag D y = eta,
// FermionicDrift.cu:57-100).  With D^dag = A + K, A = diag(2r + M + g phi) and K the
// hopping, which connects even and odd sites, the Schur complement on the even sites
//   S = A_e - K_eo A_o^-1 K_oe,   b_e = eta_e - K_eo A_o^-1 eta_o,
//   S chi_e = b_e,   chi_o = A_o^-1 (eta_o - K_oe chi_e)
// is solved by CG on S^T S chi_e = S^T b_e; S^T = A_e - H_eo A_o^-1 H_oe is the Schur
// complement of D (H = K^T, the hopping of D).  |eta - D^dag chi| = |b_e - S chi_e|
// exactly (the odd rows vanish by construction), so the solve stops on the residual of
// the unpreconditioned system, the quantity the plain solver checks.
//
// Half-lattice vectors use the compact checkerboard order of the reference's even-odd
// blocks (commented out in Dirac.cu:256-379): site (t, x) of a parity at t * Nx/2 +
// (x >> 1).  Needs even Nt and Nx.  All vectors are packed real spinors (ycn_device.hpp):
// planes [sys][c][Vh], c the spin, each entry (flavour 0, flavour 1).
//
// An iteration is one launch of the pipelined kernel (eo_pipelined.hip), in FP64 (104 B per
// site of the full lattice) or for mixed precision in FP32 (52 B), its finalize in the next
// launch's prologue or a separate kernel; mixed precision adds FP64 reliable updates whose
// residual b - S x and S^T of it take one launch of k_eo_normal_fused.  That kernel's other
// form (p' = r + beta p, v = S p', Ap = S^T v, |v|^2: four half-lattice hops through LDS) with
// the BLAS-1 update is the unpipelined FP64 iteration: where a tile of it is forced or the
// update kernel is timed.  Systems of up to 2048 even sites solve in one workgroup
// (onchip_eo.hip).
#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <type_traits>

#include "cg_fused.hpp"
#include "cg_host.hpp"
#include "pipelined.hpp"
#include "ycn_device.hpp"
#include "ycn_internal.hpp"

namespace ycn {

namespace {
constexpr int kNT = kPfNT;
}

struct EoArgs {
    int Nt, Nx, Nh, V, Vh, nNoise;   // Nh = Nx / 2, Vh = V / 2
    double r, M, g;
    int tilesX, tilesPerSys, xcdRemap;
    float invNt, invNx;              // 1 / Nt, 1 / Nx in single precision (wrapf)
    // enqueued steps (else null): the setup, drift kernels return at once while
    // *halt is set, and k_eo_eta takes its noise counter from *stepPtr
    const int *halt;
    const uint64_t *stepPtr;
};

__device__ __forceinline__ bool eo_halted(const EoArgs &A) { return A.halt && *A.halt; }

// site (t, x) of compact index j on parity par
__device__ __forceinline__ void eo_site(const EoArgs &A, int par, int j, int &t, int &x) {
    t = j / A.Nh;
    x = 2 * (j - t * A.Nh) + ((t + par) & 1);
}
__device__ __forceinline__ int eo_j(const EoArgs &A, int t, int x) { return t * A.Nh + (x >> 1); }

// Hopping (K for DAG, H otherwise) at site (t, x); ld(t', x', c) returns component c of
// the input at neighbour (t', x') of the other parity.
template <bool DAG, typename R, typename V2, typename Ld>
__device__ __forceinline__ void eo_hop(const EoArgs &A, int t, int x, Ld ld, V2 o[2]) {
    const int tp = (t == A.Nt - 1) ? 0 : t + 1, tm = (t == 0) ? A.Nt - 1 : t - 1;
    const int xp = (x == A.Nx - 1) ? 0 : x + 1, xm = (x == 0) ? A.Nx - 1 : x - 1;
    const R sf = (t == A.Nt - 1) ? (R)-1 : (R)1, sb = (t == 0) ? (R)-1 : (R)1;
    const R hp = (R)(0.5 * (A.r + 1.0)), hm = (R)(0.5 * (A.r - 1.0)), hr = (R)(0.5 * A.r), h = (R)0.5;
#pragma unroll
    for (int f = 0; f < 2; f += 2)
        hop_flavour_r<DAG, R, V2>(hp, hm, hr, h, ld(tp, x, f), ld(tp, x, f + 1), sf, ld(tm, x, f), ld(tm, x, f + 1),
                                  sb, ld(t, xp, f), ld(t, xp, f + 1), ld(t, xm, f), ld(t, xm, f + 1), o[f], o[f + 1]);
}

// ---------------------------------------------------------------------------
// setup, Schur blocks for setup and reliable updates, drift (FP64, untiled)
// ---------------------------------------------------------------------------

// eta generated (GEN) or given; u_o = A_o^-1 eta_o on the odd sites (compact layout);
// partial |eta|^2 over the full lattice
template <bool GEN>
__global__ void __launch_bounds__(kNT)
k_eo_eta(EoArgs A, const uint64_t *__restrict__ seeds, uint32_t streamBase, uint64_t step, const double *__restrict__ phi,
         double2 *__restrict__ eta, double2 *__restrict__ u, double2 *__restrict__ part) {
    __shared__ double2 lds[kNT / kWave];
    if (eo_halted(A)) return;
    if (A.stepPtr) step = *A.stepPtr;
    const int sys = blockIdx.y, s = blockIdx.x * kNT + threadIdx.x;
    const size_t V = A.V, off = (size_t)sys * 2 * V;
    double2 acc = make_double2(0.0, 0.0);
    if (s < A.V) {
        double2 b[2];
        if (GEN) {
            eta_planes<2>(seeds, streamBase, step, sys, A.nNoise, s, b);
#pragma unroll
            for (int c = 0; c < 2; ++c) eta[off + c * V + s] = b[c];
        } else {
#pragma unroll
            for (int c = 0; c < 2; ++c) b[c] = eta[off + c * V + s];
        }
#pragma unroll
        for (int c = 0; c < 2; ++c) acc.x += b[c].x * b[c].x + b[c].y * b[c].y;
        const int t = s / A.Nx, x = s - t * A.Nx;
        if ((t + x) & 1) {
            const double inv = 1.0 / (2.0 * A.r + A.M + A.g * phi[(size_t)(sys / A.nNoise) * V + s]);
            const size_t j = (size_t)sys * 2 * A.Vh + eo_j(A, t, x);
#pragma unroll
            for (int c = 0; c < 2; ++c) u[j + (size_t)c * A.Vh] = make_double2(b[c].x * inv, b[c].y * inv);
        }
    }
    acc = block_sum2<kNT>(acc, lds);
    if (threadIdx.x == 0) part[(size_t)sys * gridDim.x + blockIdx.x] = acc;
}

// b_e = eta_e - K_eo u_o with u_o = A_o^-1 eta_o (from k_eo_eta)
__global__ void __launch_bounds__(kNT)
k_eo_rhs(EoArgs A, const double2 *__restrict__ eta, const double2 *__restrict__ u, double2 *__restrict__ b) {
    if (eo_halted(A)) return;
    const int sys = blockIdx.y, j = blockIdx.x * kNT + threadIdx.x;
    if (j >= A.Vh) return;
    int t, x;
    eo_site(A, 0, j, t, x);
    const size_t V = A.V, Vh = A.Vh;
    const double2 *e = eta + (size_t)sys * 2 * V;
    const double2 *uo = u + (size_t)sys * 2 * Vh;
    double2 k[2];
    eo_hop<true, double, double2>(A, t, x, [&](int tn, int xn, int c) { return uo[c * Vh + eo_j(A, tn, xn)]; }, k);
    const size_t fs = (size_t)t * A.Nx + x;
    double2 *bo = b + (size_t)sys * 2 * Vh;
#pragma unroll
    for (int c = 0; c < 2; ++c) bo[c * Vh + j] = csub(e[c * V + fs], k[c]);
}

// U_o = A_o^-1 K_oe in_e (DAG) or A_o^-1 H_oe in_e
template <bool DAG>
__global__ void __launch_bounds__(kNT)
k_eo_hop_oe(EoArgs A, const double *__restrict__ phi, const double2 *__restrict__ in, double2 *__restrict__ U) {
    if (eo_halted(A)) return;
    const int sys = blockIdx.y, j = blockIdx.x * kNT + threadIdx.x;
    if (j >= A.Vh) return;
    int t, x;
    eo_site(A, 1, j, t, x);
    const size_t Vh = A.Vh, off = (size_t)sys * 2 * Vh;
    const double *ph = phi + (size_t)(sys / A.nNoise) * A.V;
    double2 k[2];
    eo_hop<DAG, double, double2>(A, t, x, [&](int tn, int xn, int c) { return in[off + c * Vh + eo_j(A, tn, xn)]; },
                                 k);
    const double inv = 1.0 / (2.0 * A.r + A.M + A.g * ph[(size_t)t * A.Nx + x]);
#pragma unroll
    for (int c = 0; c < 2; ++c) U[off + c * Vh + j] = make_double2(k[c].x * inv, k[c].y * inv);
}

// half-lattice vectors a setup launch also clears at its sites (any may be null)
struct EoZero {
    double2 *d[3];
    float2 *f[3];
};

// v_e = A_e in_e - K_eo U_o (DAG: S in) or A_e in_e - H_eo U_o (S^T in).
// MODE 0: out = v; MODE 1: out = b - v and partial |out|^2; MODE 2 (a solve's setup):
// out = v and partial |v|^2, and the vectors of z cleared.  out32 (optional) receives
// an FP32 copy of out.
template <bool DAG, int MODE>
__global__ void __launch_bounds__(kNT)
k_eo_hop_eo(EoArgs A, const double *__restrict__ phi, const double2 *__restrict__ in, const double2 *__restrict__ U,
            const double2 *__restrict__ b, double2 *__restrict__ out, float2 *__restrict__ out32,
            double2 *__restrict__ part, EoZero z) {
    __shared__ double2 lds[kNT / kWave];
    if (eo_halted(A)) return;
    const int sys = blockIdx.y, j = blockIdx.x * kNT + threadIdx.x;
    const size_t Vh = A.Vh, off = (size_t)sys * 2 * Vh;
    double2 acc = make_double2(0.0, 0.0);
    if (j < A.Vh) {
        int t, x;
        eo_site(A, 0, j, t, x);
        const double *ph = phi + (size_t)(sys / A.nNoise) * A.V;
        double2 k[2];
        eo_hop<DAG, double, double2>(A, t, x, [&](int tn, int xn, int c) { return U[off + c * Vh + eo_j(A, tn, xn)]; },
                                     k);
        const double d = 2.0 * A.r + A.M + A.g * ph[(size_t)t * A.Nx + x];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const double2 iv = in[off + c * Vh + j];
            double2 v = make_double2(d * iv.x - k[c].x, d * iv.y - k[c].y);
            if (MODE == 1) v = csub(b[off + c * Vh + j], v);
            out[off + c * Vh + j] = v;
            if (out32) out32[off + c * Vh + j] = make_float2((float)v.x, (float)v.y);
            acc.x += v.x * v.x + v.y * v.y;
            if (MODE == 2) {
#pragma unroll
                for (int q = 0; q < 3; ++q) {
                    if (z.d[q]) z.d[q][off + c * Vh + j] = make_double2(0.0, 0.0);
                    if (z.f[q]) z.f[q][off + c * Vh + j] = make_float2(0.f, 0.f);
                }
            }
        }
    }
    if (MODE != 0) {
        acc = block_sum2<kNT>(acc, lds);
        if (threadIdx.x == 0) part[(size_t)sys * gridDim.x + blockIdx.x] = acc;
    }
}

// drift_x = fac Re sum_k conj(chi_xk) eta_xk (FermionicDrift.cu:83-100) with chi_e from
// the solve and chi_o = A_o^-1 (eta_o - K_oe chi_e) formed on the fly; mean over noise
// vectors.
__global__ void __launch_bounds__(kNT)
k_eo_drift(EoArgs A, const double *__restrict__ phi, const double2 *__restrict__ chi_e,
           const double2 *__restrict__ eta, double *__restrict__ drift, double fac) {
    if (eo_halted(A)) return;
    const int s = blockIdx.x * kNT + threadIdx.x;
    if (s >= A.V) return;
    const int rep = blockIdx.y;
    const size_t V = A.V, Vh = A.Vh;
    const int t = s / A.Nx, x = s - t * A.Nx;
    const double *ph = phi + (size_t)rep * V;
    const bool odd = ((t + x) & 1) != 0;
    const double d = 2.0 * A.r + A.M + A.g * ph[s];
    double acc = 0.0;
    for (int jn = 0; jn < A.nNoise; ++jn) {
        const size_t sys = (size_t)rep * A.nNoise + jn;
        const double2 *ce = chi_e + sys * 2 * Vh;
        const double2 *e = eta + sys * 2 * V;
        double2 ch[2];
        if (odd) {
            double2 k[2];
            eo_hop<true, double, double2>(A, t, x, [&](int tn, int xn, int c) { return ce[c * Vh + eo_j(A, tn, xn)]; },
                                          k);
            const double inv = 1.0 / d;
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const double2 ev = e[c * V + s];
                ch[c] = make_double2((ev.x - k[c].x) * inv, (ev.y - k[c].y) * inv);
            }
        } else {
#pragma unroll
            for (int c = 0; c < 2; ++c) ch[c] = ce[c * Vh + eo_j(A, t, x)];
        }
        const double2 e0 = e[s], e1 = e[V + s];
        acc += (ch[0].x * e0.x + ch[0].y * e0.y) + (ch[1].x * e1.x + ch[1].y * e1.y);
    }
    drift[(size_t)rep * V + s] = (A.nNoise == 1) ? fac * acc : fac * acc / (double)A.nNoise;
}

// gamma_5 = sigma_2 on each flavour's spin pair, (c0, c1) -> (-i c1, i c0); with it
// gamma_5 D gamma_5 = D^dag for the Wilson-Yukawa operator (Dirac.cu:144-190).  For a real
// source gamma_5 src = i (-c1, c0): the solve runs on the real spinor (-c1, c0), and since
// gamma_5 i (a0, a1) = (a1, -a0) the result is real too.

// v = -i gamma_5 v in place (system 0): (c0, c1) -> (-c1, c0)
__global__ void __launch_bounds__(kNT) k_g5(int V, double2 *__restrict__ v) {
    const int s = blockIdx.x * kNT + threadIdx.x;
    if (s >= V) return;
    const double2 a = v[s], b = v[V + s];
    v[s] = make_double2(-b.x, -b.y);
    v[V + s] = a;
}

// The measurement's propagator from the even-odd solve of D^dag chi = eta with
// eta = -i gamma_5 src (system 0): chi on both parities (the odd sites rebuilt as in
// k_eo_drift) and out = gamma_5 i chi = D^-1 src, full lattice, packed.
__global__ void __launch_bounds__(kNT)
k_eo_propagator(EoArgs A, const double *__restrict__ phi, const double2 *__restrict__ chi_e,
                const double2 *__restrict__ eta, double2 *__restrict__ out) {
    const int s = blockIdx.x * kNT + threadIdx.x;
    if (s >= A.V) return;
    const size_t V = A.V, Vh = A.Vh;
    const int t = s / A.Nx, x = s - t * A.Nx;
    double2 ch[2];
    if ((t + x) & 1) {
        double2 k[2];
        eo_hop<true, double, double2>(A, t, x, [&](int tn, int xn, int c) { return chi_e[c * Vh + eo_j(A, tn, xn)]; },
                                      k);
        const double inv = 1.0 / (2.0 * A.r + A.M + A.g * phi[s]);
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const double2 ev = eta[c * V + s];
            ch[c] = make_double2((ev.x - k[c].x) * inv, (ev.y - k[c].y) * inv);
        }
    } else {
#pragma unroll
        for (int c = 0; c < 2; ++c) ch[c] = chi_e[c * Vh + eo_j(A, t, x)];
    }
    out[s] = ch[1];
    out[V + s] = make_double2(-ch[0].x, -ch[0].y);
}

// ---------------------------------------------------------------------------
// finalize kernels (one block per system, fixed-order sums)
// ---------------------------------------------------------------------------
// |eta|^2 and |c|^2 = |S^T b|^2: rr, thresholds and run flags of a new solve
__global__ void __launch_bounds__(kNT)
k_fin_eo_setup(const double2 *__restrict__ partE, int nbE, const double2 *__restrict__ partC, int nbC,
               CgState *__restrict__ st, int *__restrict__ active, double tol, int mode, int maxIter, int maxRestarts,
               double stopScale, const StepCtl *__restrict__ ctl) {
    __shared__ double2 lds0[kNT / kWave], lds1[kNT / kWave];
    if (ctl) {   // enqueued step: nothing while halted; the threshold learned on the device
        if (ctl->halt) return;
        stopScale = ctl->stopScale;
    }
    const int sys = blockIdx.x;
    const double2 e = pf_fin_sum(partE + (size_t)sys * nbE, nbE, lds0);
    const double2 cc = pf_fin_sum(partC + (size_t)sys * nbC, nbC, lds1);
    if (threadIdx.x) return;
    CgState &S = st[sys];
    S.enorm2 = e.x;
    S.rr = cc.x;
    S.rr_prev = cc.x;
    S.rrRel = cc.x;
    S.bnorm2 = cc.x;
    S.tol = tol;
    S.mode = mode;
    S.maxIter = maxIter;
    S.maxRestarts = maxRestarts;
    S.stop0 = (mode == YCN_TOL_ABS_RECURSIVE) ? tol : tol * sqrt(cc.x);
    S.stop = (mode == YCN_TOL_REL_TRUE) ? S.stop0 * stopScale : S.stop0;
    S.need = 0.0;
    S.nRu = 0;
    S.beta = 0.0;
    S.alpha = make_double2(0.0, 0.0);
    S.iter = 0;
    S.iter0 = 0;
    S.even = 1;
    S.pfBase = 0;
    S.pfLaunch = 0;
    S.restarts = 0;
    S.true_rel = 0.0;
    S.rz = 0.0;
    S.true_prev = 1.0;
    S.precOff = 0;
    S.restartNext = 0;
    const bool run = (0 < maxIter) && (sqrt(cc.x) > S.stop);
    S.done = run ? 0 : 1;
    S.final_ = run ? 0 : 1;
    S.converged = run ? 0 : 1;
    if (!run) atomicSub(active, 1);
}

// FP64 solve: true residual |b_e - S x_e| / |eta|.  While it exceeds tol (relative mode)
// the iteration continues from its current state with the normal-equation threshold
// lowered by the missing factor (times 1/2).
__global__ void __launch_bounds__(kNT)
k_fin_eo_true(const double2 *__restrict__ part, int nb, CgState *__restrict__ st, int *__restrict__ active) {
    __shared__ double2 lds[kNT / kWave];
    const int sys = blockIdx.x;
    const double2 tot = pf_fin_sum(part + (size_t)sys * nb, nb, lds);
    if (threadIdx.x) return;
    CgState &S = st[sys];
    S.true_rel = S.enorm2 > 0.0 ? sqrt(tot.x / S.enorm2) : sqrt(tot.x);
    S.pfLaunch = 0;
    if (S.mode != YCN_TOL_REL_TRUE) return;
    if (S.done && S.true_rel > 0.0) S.need = sqrt(S.rr) * S.tol / S.true_rel;   // paused at the stop
    if (S.true_rel > S.tol && S.iter < S.maxIter && S.restarts < S.maxRestarts) {
        S.restarts += 1;
        S.stop = sqrt(S.rr) * 0.5 * S.tol / S.true_rel;
        S.converged = 0;
        S.iter0 = S.iter;
        S.pfBase = S.iter;
        if (S.done) {
            S.done = 0;
            atomicAdd(active, 1);
        }
    } else {
        S.converged = S.true_rel <= S.tol ? 1 : 0;
    }
}

// ---------------------------------------------------------------------------
// fused Schur normal operator: p' = r + beta p_old; v = S p'; Ap = S^T v; |v|^2
// ---------------------------------------------------------------------------
// One block owns a TT x TX tile of the full lattice (TT, TX even) and produces Ap on the
// tile's TT*TX/2 even sites.  LDS holds the tile plus a 4-site halo, (TT+8) x (TX+8)
// sites in full-lattice coordinates, split by lattice parity: E[c][row][k] and
// O[c][row][k] hold the site of that parity in array row `row`, column 2k or 2k+1
// (k = column >> 1), two planes (spins) each.  Lanes of a wave take consecutive k, so every
// neighbour read (rows row +- 1 at the same k, the same row at k or k +- 1) is a
// contiguous run: no bank conflicts.  Each stage fills the parity it produces on a halo
// one site smaller than the stage before:
//   0: p'  on even sites, 4-site halo (from HBM/L2; p' of the tile also written out)
//   1: U = K p' / d on odd sites, 3-site halo          (= A_o^-1 K_oe p')
//   2: v = d p' - K U on even sites, 2-site halo        (= S p', overwrites p')
//   3: W = H v / d on odd sites, 1-site halo            (overwrites U)
//   4: Ap = d v - H W on the tile's even sites          (= S^T S p')
// The diagonal d = 2r + M + g phi is staged per parity for the whole array.  |v|^2 over
// the tile (= <p', Ap>) is the block's partial.  HBM traffic per launch: read r, p_old
// (Vh sites each) and phi, write p', Ap: 4 S/2 + P per site of the full lattice (S = 32 B in FP64).
constexpr int eo_threads(int tt, int tx) { return (tt * tx / 2 < kWave) ? kWave : tt * tx / 2; }

// RU = true: the reliable update's residual instead of an iteration.  Stage 0 stages x (r holds
// x, beta = 0), stage 2 forms res = b - S x with b (Ap_in) read at its own sites, stage 4 writes
// r = S^T res (Ap) and its FP32 copy (out32); the partials are |res|^2 (part) and |r|^2 (part2).
// Systems already final are skipped.
// WR1 = true: Wilson parameter r = 1 (hop_flavour_r1), chosen at launch when A.r == 1.
template <int TT, int TX, bool RU, bool WR1>
__global__ void __launch_bounds__(eo_threads(TT, TX))
k_eo_normal_fused(EoArgs A, const double *__restrict__ phi, CgState *st, const double2 *__restrict__ r,
                  const double2 *__restrict__ Ap_in, const double2 *__restrict__ pold, double2 *__restrict__ pnew,
                  double2 *__restrict__ Ap, double2 *__restrict__ part, float2 *__restrict__ out32,
                  double2 *__restrict__ part2) {
    using R = double;
    using V2 = double2;
    constexpr int H = TT + 8, K = (TX + 8) / 2, NT = eo_threads(TT, TX);
    constexpr int M0 = (H * K + NT - 1) / NT;
    // O and FO hold only array rows 1 .. H - 2 (odd sites are needed on the 3-site halo at
    // most): odd-site entry (row, k) sits at (row - 1) K + k, 7-8 % less LDS per block
    constexpr int HO = H - 2;
    __shared__ V2 E[2][H * K];
    __shared__ V2 O[2][HO * K];
    __shared__ R FE[H * K], FO[HO * K];
    __shared__ double2 red[NT / kWave > 0 ? NT / kWave : 1];

    const int sys = blockIdx.y;
    if (RU ? st[sys].final_ : st[sys].done) return;
    const int nTiles = A.tilesPerSys;
    const int Nt = A.Nt, Nx = A.Nx, Nh = A.Nh;
    const unsigned Vh = (unsigned)A.Vh;
    const size_t off = (size_t)sys * 2 * A.Vh;   // this system's vectors
    r += off;
    if (!RU) {
        pold += off;
        pnew += off;
    }
    Ap += off;
    if (RU) Ap_in += off;
    if (RU) out32 += off;
    const R beta = RU ? (R)0 : (R)st[sys].beta;
    const R *ph = phi + (size_t)(sys / A.nNoise) * A.V;
    const R hp = (R)(0.5 * (A.r + 1.0)), hm = (R)(0.5 * (A.r - 1.0)), hr = (R)(0.5 * A.r), h = (R)0.5;
    const R d0 = (R)(2.0 * A.r + A.M), g = (R)A.g;

    // tile origin of tile number t (contiguous bands of tiles per XCD)
    auto origin = [&](int t, int &t0, int &x0) {
        if (A.xcdRemap) t = (t % 8) * (nTiles / 8) + t / 8;
        const int ty = t / A.tilesX, tx = t - ty * A.tilesX;
        t0 = ty * TT;
        x0 = tx * TX;
    };

    // stage-0 inputs of one tile, loaded into registers: a thread handles M0 sites of the
    // array's even sites.  Array (row, col) is lattice site (t0 - 4 + row, x0 - 4 + col);
    // its parity is (row + col) & 1 because t0 + x0 is even.
    struct Regs {
        V2 ra[M0][2], pa[M0][2];
        R fe[M0], fo[M0];
        unsigned jj[M0];
    };
    auto load0 = [&](int t0, int x0, Regs &G) {
#pragma unroll
        for (int u = 0; u < M0; ++u) {
            const int w = threadIdx.x + u * NT;
            if (w < H * K) {
                const int row = w / K, k = w - row * K;
                const int gt = wrapf(t0 - 4 + row, Nt, A.invNt);
                const int colE = 2 * k + (row & 1), colO = 2 * k + 1 - (row & 1);
                const int gxE = wrapf(x0 - 4 + colE, Nx, A.invNx), gxO = wrapf(x0 - 4 + colO, Nx, A.invNx);
                G.jj[u] = (unsigned)(gt * Nh + (gxE >> 1));
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const unsigned i = c * Vh + G.jj[u];
                    G.ra[u][c] = at(r, i);
                    if (!RU) G.pa[u][c] = at(pold, i);
                }
                G.fe[u] = at(ph, (unsigned)(gt * Nx + gxE));
                G.fo[u] = at(ph, (unsigned)(gt * Nx + gxO));
            }
        }
    };
    // stage 0 proper: p' into LDS and, on the tile, to global memory; d on both parities
    auto compute0 = [&](const Regs &G) {
#pragma unroll
        for (int u = 0; u < M0; ++u) {
            const int w = threadIdx.x + u * NT;
            if (w < H * K) {
                const int row = w / K, k = w - row * K;
                const int colE = 2 * k + (row & 1);
                const bool inner = row >= 4 && row < 4 + TT && colE >= 4 && colE < 4 + TX;
#pragma unroll
                for (int c = 0; c < 2; ++c) {
                    const V2 a = G.ra[u][c];
                    const V2 pv = RU ? a : mk2<R>(a.x + beta * G.pa[u][c].x, a.y + beta * G.pa[u][c].y);
                    E[c][w] = pv;
                    if (inner && !RU) at(pnew, c * Vh + G.jj[u]) = pv;
                }
                FE[w] = d0 + g * G.fe[u];
                if (row >= 1 && row <= HO) FO[w - K] = d0 + g * G.fo[u];
            }
        }
    };

    // the sites of parity `par` in rows/cols [4 - hh, 4 + T + hh): w -> (row, k) and the
    // array indices of the site and its four neighbours (other parity)
    struct Site {
        int row, col, i, itf, itb, ixf, ixb;
    };
    auto site_of = [](int w, int hh, int par) {
        constexpr int Kw = K;
        const int c0 = 4 - hh, half = (TX + 2 * hh) / 2;
        Site q;
        q.row = c0 + w / half;
        q.col = c0 + 2 * (w - (q.row - c0) * half) + (((par + q.row) ^ c0) & 1);
        const int k = q.col >> 1;
        q.i = q.row * Kw + k;
        q.itf = q.i + Kw;
        q.itb = q.i - Kw;
        q.ixf = q.row * Kw + ((q.col + 1) >> 1);
        q.ixb = q.row * Kw + ((q.col - 1) >> 1);
        return q;
    };

    double acc = 0.0, nu = 0.0;
    // stages 1-4 of the tile at (t0, x0); stage 0 must be in LDS
    auto stages = [&](int t0, int x0) {
        // hopping at site q from the other-parity array N (component stride NS, entries
        // shifted down by SH: 0 for E, K for O)
        auto hop_at = [&](auto dag, auto ns, auto sh, const Site &q, const V2 *N, V2 o[2]) {
            constexpr bool DAG = decltype(dag)::value;
            constexpr int NS = decltype(ns)::value, SH = decltype(sh)::value;
            const int gt = wrapf(t0 - 4 + q.row, Nt, A.invNt);
            const R sf = (gt == Nt - 1) ? (R)-1 : (R)1, sb = (gt == 0) ? (R)-1 : (R)1;
            const int itf = q.itf - SH, itb = q.itb - SH, ixf = q.ixf - SH, ixb = q.ixb - SH;
#pragma unroll
            for (int f = 0; f < 2; f += 2) {
                const V2 *N0 = N + f * NS, *N1 = N + (f + 1) * NS;
                if constexpr (WR1)
                    hop_flavour_r1<DAG, R, V2>(N0[itf], N1[itf], sf, N0[itb], N1[itb], sb, N0[ixf], N1[ixf], N0[ixb],
                                               N1[ixb], o[f], o[f + 1]);
                else
                    hop_flavour_r<DAG, R, V2>(hp, hm, hr, h, N0[itf], N1[itf], sf, N0[itb], N1[itb], sb, N0[ixf],
                                              N1[ixf], N0[ixb], N1[ixb], o[f], o[f + 1]);
            }
        };
        using FromE = std::integral_constant<int, H * K>;
        using FromO = std::integral_constant<int, HO * K>;
        using Sh0 = std::integral_constant<int, 0>;
        using ShK = std::integral_constant<int, K>;
        // stage 1: U = K p' / d on odd sites, 3-site halo
        for (int w = threadIdx.x; w < (TT + 6) * ((TX + 6) / 2); w += NT) {
            const Site q = site_of(w, 3, 1);
            V2 o[2];
            hop_at(std::true_type(), FromE(), Sh0(), q, &E[0][0], o);
            const R inv = (R)1 / FO[q.i - K];
#pragma unroll
            for (int c = 0; c < 2; ++c) O[c][q.i - K] = mk2<R>(o[c].x * inv, o[c].y * inv);
        }
        __syncthreads();
        // stage 2: v = d p' - K U on even sites, 2-site halo; |v|^2 over the tile
        for (int w = threadIdx.x; w < (TT + 4) * ((TX + 4) / 2); w += NT) {
            const Site q = site_of(w, 2, 0);
            V2 o[2];
            hop_at(std::true_type(), FromO(), ShK(), q, &O[0][0], o);
            const R d = FE[q.i];
            const bool inner = q.row >= 4 && q.row < 4 + TT && q.col >= 4 && q.col < 4 + TX;
            unsigned jb = 0;   // RU: this site's entry of b
            if (RU)
                jb = (unsigned)(wrapf(t0 - 4 + q.row, Nt, A.invNt) * Nh + (wrapf(x0 - 4 + q.col, Nx, A.invNx) >> 1));
            R vs = 0;
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const V2 pv = E[c][q.i];
                V2 v = mk2<R>(d * pv.x - o[c].x, d * pv.y - o[c].y);
                if (RU) {
                    const V2 bb = at(Ap_in, c * Vh + jb);
                    v = mk2<R>(bb.x - v.x, bb.y - v.y);
                }
                E[c][q.i] = v;
                vs += v.x * v.x + v.y * v.y;
            }
            if (inner) acc += (double)vs;
        }
        __syncthreads();
        // stage 3: W = H v / d on odd sites, 1-site halo
        for (int w = threadIdx.x; w < (TT + 2) * ((TX + 2) / 2); w += NT) {
            const Site q = site_of(w, 1, 1);
            V2 o[2];
            hop_at(std::false_type(), FromE(), Sh0(), q, &E[0][0], o);
            const R inv = (R)1 / FO[q.i - K];
#pragma unroll
            for (int c = 0; c < 2; ++c) O[c][q.i - K] = mk2<R>(o[c].x * inv, o[c].y * inv);
        }
        __syncthreads();
        // stage 4: Ap = d v - H W on the tile's even sites (RU: and |r|^2)
        for (int w = threadIdx.x; w < TT * (TX / 2); w += NT) {
            const Site q = site_of(w, 0, 0);
            V2 o[2];
            hop_at(std::false_type(), FromO(), ShK(), q, &O[0][0], o);
            const R d = FE[q.i];
            // stage-4 sites are the tile's own: no wrap
            const unsigned j = (unsigned)((t0 - 4 + q.row) * Nh + ((x0 - 4 + q.col) >> 1));
            R as = 0;
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const V2 v = E[c][q.i];
                const V2 a = mk2<R>(d * v.x - o[c].x, d * v.y - o[c].y);
                at(Ap, c * Vh + j) = a;
                if (RU) at(out32, c * Vh + j) = make_float2((float)a.x, (float)a.y);
                as += a.x * a.x + a.y * a.y;
            }
            if (RU) nu += (double)as;
        }
    };

    Regs G;
    int t0, x0;
    origin(blockIdx.x, t0, x0);
    load0(t0, x0, G);
    compute0(G);
    __syncthreads();
    stages(t0, x0);
    const size_t pidx = (size_t)sys * gridDim.x + blockIdx.x;
    const double2 tot = block_sum2<NT>(make_double2(acc, RU ? nu : 0.0), red);
    if (threadIdx.x == 0) {
        part[pidx] = make_double2(tot.x, 0.0);
        if (RU) part2[pidx] = make_double2(tot.y, 0.0);
    }
}

// enqueued Langevin steps: start of a step.  The count of active systems of its
// solve, and the halt flag and counter the step's coloured noise reads, copied into a
// second block (noise): the noise runs on a branch of the graph beside the solve, whose
// check kernel may change the first block while the noise kernels run.
__global__ void k_step_begin(const StepCtl *__restrict__ ctl, StepCtl *__restrict__ noise, int *__restrict__ active,
                             int nsys) {
    if (threadIdx.x) return;
    if (!ctl->halt) *active = nsys;
    noise->halt = ctl->halt;
    noise->step = ctl->step;
}

// enqueued Langevin steps: after the step's chunk schedule.  Every system final:
// the step's statistics into the control block, the next solve's starting threshold
// (relative mode: 0.9 times the largest ratio need / stop0 the systems reported, as
// eo_learn_stop_scale does on the host) and the next step's counter.  A system still
// iterating halts the run at this step: the drift, the update and every later step's
// kernels outside the chunk schedule return at once.
__global__ void k_step_check(StepCtl *__restrict__ ctl, const CgState *__restrict__ st, int nsys, int relMode) {
    if (threadIdx.x || ctl->halt) return;
    int itMax = -1, kMax = 0, rsMax = 0, conv = 1;
    double itSum = 0.0, rrMax = 0.0, trMax = 0.0, ratio = 0.0;
    for (int k = 0; k < nsys; ++k) {
        const CgState &S = st[k];
        if (!S.final_) {
            ctl->halt = 1;
            ctl->haltStep = ctl->step;
            return;
        }
        if (S.iter > itMax) {
            itMax = S.iter;
            kMax = k;
        }
        rsMax = max(rsMax, S.restarts);
        conv &= S.converged;
        itSum += S.iter;
        rrMax = fmax(rrMax, S.rr);
        trMax = fmax(trMax, S.true_rel);
        if (S.need > 0.0 && S.stop0 > 0.0) ratio = fmax(ratio, S.need / S.stop0);
    }
    ctl->itersMaxSum += itMax;
    ctl->itersMeanSum += itSum / nsys;
    ctl->restarts += rsMax;
    ctl->converged &= conv;
    ctl->rrMax = fmax(ctl->rrMax, rrMax);
    ctl->trueRelMax = fmax(ctl->trueRelMax, trMax);
    ctl->lastIters = itMax;
    ctl->nRounds = min(st[kMax].nRu, kMaxRounds);
    for (int i = 0; i < ctl->nRounds; ++i) ctl->rounds[i] = st[kMax].ruIter[i];
    if (relMode && ratio > 0.0) ctl->stopScale = fmin(1.0, fmax(1e-3, 0.9 * ratio));
    ctl->steps += 1;
    ctl->step += 1;
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// at least 64 sites per tile: the partials buffer holds 2 V/64 entries per system.
// FP32 entries with persist = true launch only the resident blocks, each walking several
// tiles with the next tile's loads in flight.
struct EoTileCfg {
    int TT, TX;
    bool persist;
};
constexpr EoTileCfg kEoTiles64[] = {{8, 32, false}, {16, 16, false}, {4, 64, false}, {4, 32, false}, {2, 32, false}};
constexpr EoTileCfg kEoTiles32[] = {{8, 32, false},  {16, 32, false}, {8, 64, false},  {16, 16, false},
                                    {4, 64, false},  {2, 32, false},  {32, 32, false}, {16, 64, false},
                                    {8, 32, true},   {16, 32, true},  {16, 16, true},  {8, 64, true},
                                    {64, 64, false}, {32, 128, false}};
// tiles of the pipelined FP64 iteration
struct EoTile {
    int TT, TX;
};
constexpr EoTile kEoTilesP64[] = {{8, 32}, {16, 32}, {16, 16}, {4, 32}, {2, 32}, {4, 16}, {32, 32}};
constexpr int kNumEoP64 = sizeof(kEoTilesP64) / sizeof(kEoTilesP64[0]);
constexpr int kNumEo64 = sizeof(kEoTiles64) / sizeof(kEoTiles64[0]);
constexpr int kNumEo32 = sizeof(kEoTiles32) / sizeof(kEoTiles32[0]);

static EoArgs eo_args(const Ctx &c, int TT, int TX) {
    EoArgs A;
    A.Nt = c.p.Nt;
    A.Nx = c.p.Nx;
    A.Nh = c.p.Nx / 2;
    A.V = c.V;
    A.Vh = c.V / 2;
    A.nNoise = c.nNoise;
    A.r = c.p.r;
    A.M = c.p.M;
    A.g = c.p.g;
    A.tilesX = TX > 0 ? c.p.Nx / TX : 0;
    A.tilesPerSys = (TT > 0 && TX > 0) ? (c.p.Nt / TT) * (c.p.Nx / TX) : 0;
    A.xcdRemap = (A.tilesPerSys % 8 == 0) ? 1 : 0;
    A.invNt = 1.0f / (float)A.Nt;
    A.invNx = 1.0f / (float)A.Nx;
    A.halt = nullptr;
    A.stepPtr = nullptr;
    return A;
}

template <typename Tile>
static bool eo_fits(const Ctx &c, Tile t) { return c.p.Nt % t.TT == 0 && c.p.Nx % t.TX == 0; }

// the two partial slots of prologue-finalized launches (launch idx writes slot idx & 1
// and reads the other), sized for the smallest tile (64 sites: at most V / 64 blocks)
int eo_pf_alloc(Ctx &c) {
    const size_t n = (size_t)c.nSys * ((c.V + 63) / 64) * 2;
    for (double2 *&slot : c.pfSlot) {
        YCN_HIP(hipMalloc(&slot, sizeof(double2) * n));
        YCN_HIP(hipMemset(slot, 0, sizeof(double2) * n));
    }
    return YCN_OK;
}

// even extents; the fused kernels address one system's FP64 half-lattice planes and
// phi through 32-bit byte offsets and wrap halo coordinates with wrapf
// (|a| < 2^22)
static bool eo_shape_ok(const Ctx &c) {
    return c.p.Nt % 2 == 0 && c.p.Nx % 2 == 0 && c.V < (1 << 27) &&
           c.p.Nt < (1 << 21) && c.p.Nx < (1 << 21);
}

bool eo_available(const Ctx &c) { return eo_shape_ok(c) && c.tileEo64 >= 0; }

// launch the fused Schur normal operator (FP64) with tile `ti`; returns the partial count
template <int TT, int TX>
static void launch_eo_tt(const Ctx &c, int nsys, const EoArgs &A, const double *phi, const double2 *r,
                         const double2 *pold, double2 *pnew, double2 *Ap) {
    auto *k = A.r == 1.0 ? &k_eo_normal_fused<TT, TX, false, true> : &k_eo_normal_fused<TT, TX, false, false>;
    hipLaunchKernelGGL(k, dim3(A.tilesPerSys, nsys), dim3(eo_threads(TT, TX)), 0, c.stream, A, phi, c.cg_d, r,
                       (const double2 *)nullptr, pold, pnew, Ap, c.partials, (float2 *)nullptr, (double2 *)nullptr);
}
static int launch_eo_fused(Ctx &c, int ti, int nsys, const double *phi, const double2 *r, const double2 *pold,
                           double2 *pnew, double2 *Ap) {
    const EoTileCfg t = kEoTiles64[ti];
    const EoArgs A = eo_args(c, t.TT, t.TX);
    prof_before(c, PK_NORMAL_OP, (double)nsys * c.V * (4 * 16 + 8));
    switch (ti) {
    case 0: launch_eo_tt<8, 32>(c, nsys, A, phi, r, pold, pnew, Ap); break;
    case 1: launch_eo_tt<16, 16>(c, nsys, A, phi, r, pold, pnew, Ap); break;
    case 2: launch_eo_tt<4, 64>(c, nsys, A, phi, r, pold, pnew, Ap); break;
    case 3: launch_eo_tt<4, 32>(c, nsys, A, phi, r, pold, pnew, Ap); break;
    default: launch_eo_tt<2, 32>(c, nsys, A, phi, r, pold, pnew, Ap); break;
    }
    prof_after(c, PK_NORMAL_OP);
    return A.tilesPerSys;
}

// the reliable update's residual in one fused FP64 launch (tile of the FP64 table):
// res = b - S x, r = S^T res (FP64 and FP32 copy), partials |res|^2 and |r|^2 of the
// systems not yet final; returns the partials per system
template <int TT, int TX>
static int launch_eo_ru_tt(Ctx &c, int nsys, const EoArgs &A, const double *phi, const double2 *x, const double2 *b,
                           double2 *r, float2 *r32, double2 *partRes, double2 *partN) {
    auto *k = A.r == 1.0 ? &k_eo_normal_fused<TT, TX, true, true> : &k_eo_normal_fused<TT, TX, true, false>;
    hipLaunchKernelGGL(k, dim3(A.tilesPerSys, nsys), dim3(eo_threads(TT, TX)), 0, c.stream, A, phi, c.cg_d, x, b,
                       (const double2 *)nullptr, (double2 *)nullptr, r, partRes, r32, partN);
    return A.tilesPerSys;
}
static int launch_eo_ru(Ctx &c, int nsys, const double *phi, const double2 *x, const double2 *b, double2 *r,
                        float2 *r32, double2 *partRes, double2 *partN) {
    const EoTileCfg t = kEoTiles64[c.tileEo64];
    const EoArgs A = eo_args(c, t.TT, t.TX);
    switch (c.tileEo64) {
    case 0: return launch_eo_ru_tt<8, 32>(c, nsys, A, phi, x, b, r, r32, partRes, partN);
    case 1: return launch_eo_ru_tt<16, 16>(c, nsys, A, phi, x, b, r, r32, partRes, partN);
    case 2: return launch_eo_ru_tt<4, 64>(c, nsys, A, phi, x, b, r, r32, partRes, partN);
    case 3: return launch_eo_ru_tt<4, 32>(c, nsys, A, phi, x, b, r, r32, partRes, partN);
    default: return launch_eo_ru_tt<2, 32>(c, nsys, A, phi, x, b, r, r32, partRes, partN);
    }
}

// scratch of a solve: b_e and U_o in c.t (first and second half), the residual in c.Ap
struct EoBufs {
    double2 *b, *U, *res;
};
static EoBufs eo_bufs(Ctx &c, int nsys) {
    const size_t h = (size_t)nsys * 2 * (c.V / 2);
    return {c.t, c.t + h, c.Ap};
}

// the pipelined FP32 iteration (k_eo_pf) with tile `ti` as launch idx of a chunk (idx & 1: the Ap
// and partial-slot parity, the directions in rotation); returns the block partials per system
static int launch_eo_pf(Ctx &c, int ti, int nsys, int idx, int finMode) {
    const EoTileCfg t = kEoTiles32[ti];
    const int par = idx & 1;
    EoPfLaunch<float> b;
    b.phi = c.phis;
    b.idx = idx;
    b.form = idx == 0 ? 0 : par ? 1 : 2;
    b.finMode = finMode;
    b.persist = t.persist;
    b.part = finMode ? c.pfSlot[par] : c.partials;
    b.prevPart = c.pfSlot[par ^ 1];
    b.Ap_in = par ? c.pfA1 : c.Aps;
    b.Ap = par ? c.Aps : c.pfA1;
    b.x = c.xs;
    // direction p_k in pf_dir(c, k); launch 0 reads r, the others p_{idx-2}
    b.r = idx == 0 ? c.rs : pf_dir(c, idx - 2);
    b.pold = pf_dir(c, idx - 1);
    b.pnew = pf_dir(c, idx);
    // half-lattice FP32 vectors: read p_{idx-2} (or r), Ap, p and write p, Ap, and x_s read and
    // written in odd launches; and read phi.  The figure counts the vectors as the complex
    // spinors of the interface (16 B per site of the full lattice), as ycn_profile_end
    // documents; packed they are half that.
    prof_before(c, PK_NORMAL_OP, (double)nsys * c.V * ((par ? 7 : 5) * 16 + 4));
    const int nb = launch_eo_pf32(c, t.TT, t.TX, nsys, b);
    prof_after(c, PK_NORMAL_OP);
    return nb;
}

// FP64 direction p_k of a phase: p[0] (p_{-1}), p[1], and r, which nothing reads after launch 0
static double2 *eo_p64_dir(const Ctx &c, int k) {
    double2 *const rot[3] = {c.pv[0], c.pv[1], c.r};
    return rot[(k + 1) % 3];
}
// launch idx of a chunk of the pipelined FP64 iteration (first: of the phase's first chunk), A p
// alternating between U_o's scratch and Ap
static int launch_eo_p64(Ctx &c, int ti, int nsys, const double *phi, int idx, bool first, int finMode) {
    const EoTile t = kEoTilesP64[ti];
    const int par = idx & 1;
    double2 *const U = eo_bufs(c, nsys).U;
    EoPfLaunch<double> b;
    b.phi = phi;
    b.idx = idx;
    b.form = first && idx == 0 ? 0 : par ? 1 : 2;
    b.finMode = finMode;
    b.persist = false;
    b.part = c.pfSlot[par];
    b.prevPart = c.pfSlot[par ^ 1];
    b.Ap_in = par ? U : c.Ap;
    b.Ap = par ? c.Ap : U;
    b.x = c.x;
    b.r = first && idx == 0 ? c.r : eo_p64_dir(c, idx + 1);   // p_{idx-2}
    b.pold = eo_p64_dir(c, idx + 2);
    b.pnew = eo_p64_dir(c, idx);
    prof_before(c, PK_NORMAL_OP, (double)nsys * c.V * ((par ? 7 : 5) * 16 + 8));
    const int nb = launch_eo_pf64(c, t.TT, t.TX, nsys, b);
    prof_after(c, PK_NORMAL_OP);
    return nb;
}

static dim3 half_grid(const Ctx &c, int nsys) { return dim3((c.V / 2 + kNT - 1) / kNT, nsys); }

// Times every even-odd tile that fits (FP64, and FP32 when the mixed buffers exist) on
// the context's buffers and keeps the fastest.  The trial launches only touch CG scratch.
int eo_autotune(Ctx &c) {
    c.tileEo64 = c.tileEo32 = c.tileEoP64 = -1;
    if (!eo_shape_ok(c)) return YCN_OK;
    hipEvent_t e0, e1;
    YCN_HIP(hipEventCreate(&e0));
    YCN_HIP(hipEventCreate(&e1));
    YCN_HIP(hipMemsetAsync(c.cg_d, 0, sizeof(CgState) * c.nSys, c.stream));
    const int reps = c.V >= (1 << 16) ? 10 : 3;
    auto time_it = [&](auto launch) -> double {   // launch(k), k = 0, 1, ... (k & 1: parity)
        launch(0);
        launch(1);
        (void)hipEventRecord(e0, c.stream);
        for (int i = 0; i < reps; ++i) launch(2 + i);
        (void)hipEventRecord(e1, c.stream);
        (void)hipEventSynchronize(e1);
        float ms = 0;
        (void)hipEventElapsedTime(&ms, e0, e1);
        return 1e3 * ms / reps;
    };
    char line[96];
    const bool pfOk = c.rs && c.phis && c.pfA1 && c.pfP2 && c.pfSlot[0] && c.pfSlot[1];
    // measured times: kNumEo64 FP64 tiles, then kNumEo32 x {separate, prologue} FP32
    // pipelined iterations (1e30 where a tile does not fit); reused from an earlier
    // context of the same shape when there is one
    std::vector<double> us;
    const bool memo = tune_lookup(1, c, us) && us.size() == (size_t)(kNumEo64 + 2 * kNumEo32);
    if (!memo) {
        us.assign(kNumEo64 + 2 * kNumEo32, 1e30);
        for (int i = 0; i < kNumEo64; ++i)
            if (eo_fits(c, kEoTiles64[i]))
                us[i] = time_it([&](int k) {
                    (void)launch_eo_fused(c, i, c.nSys, c.phi[c.cur], c.r, c.pv[k & 1], c.pv[(k & 1) ^ 1], c.Ap);
                });
        if (pfOk)
            for (int i = 0; i < kNumEo32; ++i) {
                if (!eo_fits(c, kEoTiles32[i])) continue;
                us[kNumEo64 + 2 * i] =
                    time_it([&](int k) { launch_fin_pf(c, c.nSys, launch_eo_pf(c, i, c.nSys, k, 0), 0, c.partials); });
                us[kNumEo64 + 2 * i + 1] = time_it([&](int k) { (void)launch_eo_pf(c, i, c.nSys, k, 2); });
            }
        tune_store(1, c, us);
    }
    c.tuneReport += memo ? " | even-odd fp64 tiles (us/launch, measured by an earlier context):"
                         : " | even-odd fp64 tiles (us/launch):";
    double best = 1e30;
    for (int i = 0; i < kNumEo64; ++i) {
        if (!eo_fits(c, kEoTiles64[i])) continue;
        std::snprintf(line, sizeof line, " %dx%d %.1f;", kEoTiles64[i].TT, kEoTiles64[i].TX, us[i]);
        c.tuneReport += line;
        if (us[i] < best) { best = us[i]; c.tileEo64 = i; }
    }
    // FP32 pipelined iteration: each tile with the separate finalize and with the
    // finalize in the next launch's prologue; YCN_EO_FIN=separate|fused restricts the
    // choice to one form
    const char *fin = std::getenv("YCN_EO_FIN");
    const bool allowSep = !fin || std::strcmp(fin, "fused") != 0;
    const bool allowFused = !fin || std::strcmp(fin, "separate") != 0;
    double us32[kNumEo32][2] = {};
    for (int i = 0; i < kNumEo32; ++i) {
        us32[i][0] = us[kNumEo64 + 2 * i];
        us32[i][1] = us[kNumEo64 + 2 * i + 1];
    }
    if (pfOk) {
        c.tuneReport += " | even-odd fp32 pipelined tiles (us/iteration, separate | prologue finalize):";
        best = 1e30;
        for (int i = 0; i < kNumEo32; ++i) {
            if (!eo_fits(c, kEoTiles32[i])) continue;
            std::snprintf(line, sizeof line, " %dx%d%s %.1f|%.1f;", kEoTiles32[i].TT, kEoTiles32[i].TX,
                          kEoTiles32[i].persist ? "p" : "", us32[i][0], us32[i][1]);
            c.tuneReport += line;
            for (int m = 0; m < 2; ++m)
                if ((m ? allowFused : allowSep) && us32[i][m] < best) {
                    best = us32[i][m];
                    c.tileEo32 = i;
                    c.eoFinFused = m == 1;
                }
        }
    }
    // YCN_TILE_EO / YCN_TILE_EO32 force a tile of the tables (tests cover every shape)
    if (const char *f = std::getenv("YCN_TILE_EO")) {
        const int i = std::atoi(f);
        if (i >= 0 && i < kNumEo64 && eo_fits(c, kEoTiles64[i])) c.tileEo64 = i;
        c.tuneReport += " (even-odd fp64 tile forced by YCN_TILE_EO)";
    }
    if (const char *f = std::getenv("YCN_TILE_EO32")) {
        const int i = std::atoi(f);
        if (c.rs && c.phis && c.pfA1 && c.pfP2 && c.pfSlot[0] && i >= 0 && i < kNumEo32 && eo_fits(c, kEoTiles32[i])) {
            c.tileEo32 = i;
            c.eoFinFused = allowFused && (!allowSep || us32[i][1] < us32[i][0]);
        }
        c.tuneReport += " (even-odd fp32 tile forced by YCN_TILE_EO32)";
    }
    // FP64 contexts: the pipelined FP64 iteration's tiles, with either finalize
    if (c.p.cgPrecision != YCN_CG_MIXED && c.tileEo64 >= 0 && c.pfSlot[1] && !onchip_eo(c) &&
        !std::getenv("YCN_TILE_EO")) {
        const bool memoP = tune_lookup(4, c, us) && us.size() == 2 * (size_t)kNumEoP64;
        if (!memoP) {
            us.assign(2 * kNumEoP64, 1e30);
            for (int i = 0; i < kNumEoP64; ++i)
                for (int m = 0; m < 2 && eo_fits(c, kEoTilesP64[i]); ++m)
                    us[2 * i + m] = time_it([&](int k) {
                        const int nb = launch_eo_p64(c, i, c.nSys, c.phi[c.cur], k, true, m ? 2 : 0);
                        if (!m) launch_fin_p64(c, c.nSys, nb, 1, c.pfSlot[k & 1], 0);
                    });
            tune_store(4, c, us);
        }
        const char *force = std::getenv("YCN_TILE_PL");
        const int f = force ? std::atoi(force) : -1;
        best = 1e30;
        c.tuneReport += " | even-odd fp64 pipelined tiles (us/iteration, separate | prologue finalize):";
        for (int i = 0; i < kNumEoP64; ++i) {
            if (!eo_fits(c, kEoTilesP64[i])) continue;
            std::snprintf(line, sizeof line, " %dx%d %.1f|%.1f;", kEoTilesP64[i].TT, kEoTilesP64[i].TX, us[2 * i],
                          us[2 * i + 1]);
            c.tuneReport += line;
            for (int m = 0; m < 2; ++m)
                if ((f < 0 || f == i) && us[2 * i + m] < best && (m ? allowFused : allowSep)) {
                    best = us[2 * i + m];
                    c.tileEoP64 = i;
                    c.eoFinFused = m == 1;
                }
        }
    }
    if (c.tileEoP64 >= 0)
        tune_report_choice(c, "fp64", kEoTilesP64[c.tileEoP64].TT, kEoTilesP64[c.tileEoP64].TX, "");
    if (c.tileEo32 >= 0 && c.p.cgPrecision == YCN_CG_MIXED) {
        const EoTileCfg t = kEoTiles32[c.tileEo32];
        tune_report_choice(c, "fp32", t.TT, t.TX, t.persist ? "p" : "");
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    YCN_HIP(hipGetLastError());
    YCN_HIP(hipMemsetAsync(c.cg_d, 0, sizeof(CgState) * c.nSys, c.stream));
    YCN_HIP(hipStreamSynchronize(c.stream));
    return YCN_OK;
}

static void launch_eo_iteration(Ctx &c, int nsys, const double *phi, int parity) {
    const int nb = launch_eo_fused(c, c.tileEo64, nsys, phi, c.r, c.pv[parity], c.pv[parity ^ 1], c.Ap);
    launch_fin_alpha(c, nsys, nb);
    const int nbu = launch_cg_update(c, nsys, c.V / 2, c.pv[parity ^ 1]);
    launch_fin_beta(c, nsys, nbu, false, true);
}

// One captured chunk of pipelined FP64 iterations (first: of a phase, from the residual in r and the
// direction in p[0]).  A phase is what runs until every system has stopped; the close ends it.
static int eo_p64_iterations(Ctx &c, const double *phi, int nsys, bool first) {
    const bool fused = c.eoFinFused;
    return run_chunk(c, phi, nsys, YCN_DAGGER, kP64Launches, first ? 6 : 7, kPacked, c.tileEoP64, [&](int i) {
        const int nb = launch_eo_p64(c, c.tileEoP64, nsys, phi, i, first, fused ? 1 : 0);
        if (!fused || i == kP64Launches - 1)
            launch_fin_p64(c, nsys, nb, fused ? kP64Launches : 1, c.pfSlot[i & 1], 1);
    });
}

// launch i of a chunk of the pipelined FP32 iteration: one launch that finalizes its
// predecessor in the prologue, or the fused kernel and k_fin_pf (whichever the autotuner
// timed faster)
static void launch_eo_pf_iteration(Ctx &c, int nsys, int i) {
    if (c.eoFinFused) {
        c.eoPfBlocks = launch_eo_pf(c, c.tileEo32, nsys, i, 1);
        return;
    }
    launch_fin_pf(c, nsys, launch_eo_pf(c, c.tileEo32, nsys, i, 0), 1, c.partials);
}
// Relative mode: the recursive (normal-equation) residual at which the FP64 true
// residual reaches tol varies little between consecutive solves, so the next solve
// starts from 0.9 times the largest ratio need / stop0 the systems of this one reported
// (the first solve starts from tol |r_0|).  A threshold that proves too loose is
// tightened by the true-residual check as before; one too tight costs a few iterations.
void eo_learn_stop_scale(Ctx &c, int nsys) {
    if (c.p.cgTolMode != YCN_TOL_REL_TRUE) return;
    double r = 0.0;
    for (int k = 0; k < nsys; ++k)
        if (c.cg_h[k].need > 0.0 && c.cg_h[k].stop0 > 0.0) r = std::max(r, c.cg_h[k].need / c.cg_h[k].stop0);
    if (r > 0.0) c.eoStopScale = std::min(1.0, std::max(1e-3, 0.9 * r));
}

// the pipelined FP32 solve with FP64 reliable updates runs where its buffers exist
static bool eo_mixed(const Ctx &c) {
    return c.p.cgPrecision == YCN_CG_MIXED && c.tileEo32 >= 0 && c.rs && c.phis && c.pfA1 && c.pfP2 &&
           c.pfSlot[0] && c.pfSlot[1];
}

// Setup of a solve: eta (from the Philox streams when gen) and u_o = A_o^-1 eta_o,
// b_e = eta_e - K_eo u_o, r = S^T b (FP32 copy when mixed), x and the directions cleared,
// the FP32 copy of the field (mixed) and the per-system state.  ctl (an enqueued
// step, else null): every launch returns at once while ctl->halt is set, the noise
// counter is ctl->step and the starting threshold ctl->stopScale.
static int eo_setup(Ctx &c, const double *phi, int nsys, bool gen, uint32_t streamBase, uint64_t step, bool mixed,
                    const StepCtl *ctl) {
    EoArgs A = eo_args(c, 0, 0);
    if (ctl) {
        A.halt = &ctl->halt;
        A.stepPtr = &ctl->step;
    }
    const dim3 gF((c.V + kNT - 1) / kNT, nsys), gH = half_grid(c, nsys);
    const int nbF = gF.x, nbH = gH.x;
    double2 *partE = c.partials, *partH = c.partials + (size_t)nsys * nbF;
    const EoBufs B = eo_bufs(c, nsys);
    if (!ctl) {   // (an enqueued step sets the count in k_step_begin)
        const int rc = set_int(c, c.active, nsys);
        if (rc) return rc;
    }
    const int maxIter = c.p.cgMaxIter, maxRestarts = mixed ? 1 << 20 : 4;
    if (gen)
        hipLaunchKernelGGL(k_eo_eta<true>, gF, dim3(kNT), 0, c.stream, A, (const uint64_t *)c.seed_d, streamBase, step,
                           phi, c.eta, B.U, partE);
    else
        hipLaunchKernelGGL(k_eo_eta<false>, gF, dim3(kNT), 0, c.stream, A, (const uint64_t *)c.seed_d, streamBase,
                           step, phi, c.eta, B.U, partE);
    hipLaunchKernelGGL(k_eo_rhs, gH, dim3(kNT), 0, c.stream, A, (const double2 *)c.eta, (const double2 *)B.U, B.b);
    // r = S^T b (and its FP32 copy); the same launch clears x and the directions (FP64
    // solver: p[0], p[1]; mixed: x_s, p[0], Ap)
    hipLaunchKernelGGL(k_eo_hop_oe<false>, gH, dim3(kNT), 0, c.stream, A, phi, (const double2 *)B.b, B.U);
    EoZero zero{};
    zero.d[0] = c.x;
    if (mixed) {
        zero.f[0] = c.xs;
        zero.f[1] = c.ps[0];
        zero.f[2] = c.Aps;
    } else {
        zero.d[1] = c.pv[0];
        zero.d[2] = c.pv[1];
    }
    hipLaunchKernelGGL((k_eo_hop_eo<false, 2>), gH, dim3(kNT), 0, c.stream, A, phi, (const double2 *)B.b,
                       (const double2 *)B.U, (const double2 *)nullptr, c.r, mixed ? c.rs : (float2 *)nullptr, partH,
                       zero);
    if (mixed) {
        const int nrepUsed = (nsys + c.nNoise - 1) / c.nNoise;
        // an enqueued step also keeps the FP64 field its solve reads in c.phiSolve: the
        // reliable updates of a halted solve that later steps' chunks run read it there
        const int rc = to_f32_n(c, phi, c.phis, (int64_t)std::min(nrepUsed, c.nRep) * c.V,
                                ctl ? &ctl->halt : nullptr, ctl ? c.phiSolve : nullptr);
        if (rc) return rc;
    }
    hipLaunchKernelGGL(k_fin_eo_setup, dim3(nsys), dim3(kNT), 0, c.stream, (const double2 *)partE, nbF,
                       (const double2 *)partH, nbH, c.cg_d, c.active, c.p.cgTol, c.p.cgTolMode, maxIter, maxRestarts,
                       c.eoStopScale, ctl);
    YCN_HIP(hipGetLastError());
    return YCN_OK;
}

// One chunk of n pipelined FP32 iterations and the reliable update that closes it:
// x += x_s, p[0] = p[1]; res = b - S x; r = S^T res (FP64, FP32 copy into r[0]); then
// converged on the FP64 true residual, or resume.  Systems already final exit every
// kernel at once.
static int eo_mixed_chunk(Ctx &c, const double *phi, int nsys, int n, bool graphed) {
    const int Vh = c.V / 2;
    const dim3 gH = half_grid(c, nsys);
    const EoBufs B = eo_bufs(c, nsys);
    // reliable-update partials: at most V / 64 blocks per system each (smallest FP64 tile)
    double2 *partRu = c.partials, *partRu2 = c.partials + (size_t)nsys * ((c.V + 63) / 64);
    if (n & 1) {   // the pipelined launches defer x_s updates in pairs
        c.err = "internal: a chunk of the pipelined iteration has an odd number of launches";
        return YCN_ERR_INVALID;
    }
    if (graphed) {   // a whole step is enqueued or captured: the launches themselves
        for (int i = 0; i < n; ++i) launch_eo_pf_iteration(c, nsys, i);
    } else {
        const int rc = run_chunk(c, nullptr, nsys, YCN_DAGGER, n, 4, kPacked, c.tileEo32,
                                 [&](int i) { launch_eo_pf_iteration(c, nsys, i); });
        if (rc) return rc;
    }
    const PfChunkEnd end = pf_chunk_end(c, n);
    hipLaunchKernelGGL(k_pf_reliable, gH, dim3(kNT), 0, c.stream, Vh, end.n, (const CgState *)c.cg_d, c.x, c.xs,
                       (const float2 *)c.ps[1], (const float2 *)c.pfP2, c.ps[0]);
    const int nbR = launch_eo_ru(c, nsys, phi, c.x, B.b, c.r, c.rs, partRu, partRu2);
    hipLaunchKernelGGL(k_fin_pf_true, dim3(nsys), dim3(kNT), 0, c.stream, (const double2 *)partRu,
                       (const double2 *)partRu2, nbR, c.cg_d, c.active, end);
    YCN_HIP(hipGetLastError());
    return YCN_OK;
}

// The pipelined FP32 solve from the state the setup (or an unfinished enqueued solve) left,
// until every system is final; itDone: iterations already done.
static int eo_mixed_loop(Ctx &c, const double *phi, int nsys, int itDone, SolveStats *st) {
    const int rc = pf_loop(c, nsys, itDone, st, [&](int n) { return eo_mixed_chunk(c, phi, nsys, n, false); });
    if (!rc) eo_learn_stop_scale(c, nsys);
    return rc;
}

// Solve S chi_e = b_e for every system (eta from the Philox streams when gen); chi_e is
// left in c.x, eta in c.eta.  FP64 CG, or FP32 inner iterations with FP64 reliable
// updates when cgPrecision is mixed.
int eo_solve(Ctx &c, const double *phi, int nsys, bool gen, uint32_t streamBase, uint64_t step, SolveStats *st) {
    if (!eo_available(c)) {
        c.err = "even-odd preconditioning needs even Nt and Nx and a fused tile that divides the lattice";
        return YCN_ERR_UNSUPPORTED;
    }
    const bool mixed = eo_mixed(c);
    int rc = eo_setup(c, phi, nsys, gen, streamBase, step, mixed, nullptr);
    if (rc) return rc;
    if (mixed) return eo_mixed_loop(c, phi, nsys, 0, st);

    const EoArgs A = eo_args(c, 0, 0);
    const dim3 gH = half_grid(c, nsys);
    const int nbH = gH.x;
    double2 *partH = c.partials + (size_t)nsys * ((c.V + kNT - 1) / kNT);
    const EoBufs B = eo_bufs(c, nsys);
    const int maxIter = c.p.cgMaxIter, maxRestarts = 4;
    int launched = 0, active = nsys;
    int chunk = std::max(kGraphIters, std::min(c.lastIters, maxIter));
    const int hardCap = maxIter * (maxRestarts + 1) + 2 * kGraphIters;
    const bool pipelined = c.tileEoP64 >= 0 && c.profTarget != PK_CG_UPDATE;
    for (int guard = 0; guard < maxRestarts + 2; ++guard) {
        bool first = true;
        while (active > 0 && launched < hardCap) {
            const int n = std::min(chunk, hardCap - launched);
            for (int k = 0, m = pipelined ? kP64Launches : kGraphIters; k < n; k += m, launched += m) {
                if (pipelined)
                    rc = eo_p64_iterations(c, phi, nsys, first);
                else
                    rc = run_chunk(c, phi, nsys, YCN_DAGGER, kGraphIters, 3, kPacked, c.tileEo64,
                                   [&](int i) { launch_eo_iteration(c, nsys, phi, i & 1); });
                if (rc) return rc;
                first = false;
            }
            rc = poll_active(c, active);
            if (rc) return rc;
            chunk = std::max(kGraphIters, std::min(64, chunk / 2));
        }
        if (pipelined)
            hipLaunchKernelGGL(k_p64_close<true>, gH, dim3(kNT), 0, c.stream, c.V / 2, (const CgState *)c.cg_d, c.x,
                               c.pv[0], (const double2 *)c.pv[1], c.r, (const double2 *)B.U, (const double2 *)c.Ap);
        // true residual of the unpreconditioned system, |b_e - S x_e| / |eta|
        hipLaunchKernelGGL(k_eo_hop_oe<true>, gH, dim3(kNT), 0, c.stream, A, phi, (const double2 *)c.x, B.U);
        hipLaunchKernelGGL((k_eo_hop_eo<true, 1>), gH, dim3(kNT), 0, c.stream, A, phi, (const double2 *)c.x,
                           (const double2 *)B.U, (const double2 *)B.b, B.res, (float2 *)nullptr, partH, EoZero{});
        hipLaunchKernelGGL(k_fin_eo_true, dim3(nsys), dim3(kNT), 0, c.stream, (const double2 *)partH, nbH, c.cg_d,
                           c.active);
        YCN_HIP(hipGetLastError());
        rc = poll_active(c, active);
        if (rc) return rc;
        if (active == 0 || launched >= hardCap) break;
        chunk = kGraphIters;
    }
    rc = read_stats(c, nsys, st);
    if (rc) return rc;
    eo_learn_stop_scale(c, nsys);
    return YCN_OK;
}

// D^-1 src for the measurement's point source (src in c.eta, system 0, c.nNoise = 1):
// gamma_5 D gamma_5 = D^dag, so D^-1 src = gamma_5 (D^dag)^-1 (gamma_5 src), and the
// fermion-force solve of D^dag chi = eta gives it.  The solve's iteration count, starting
// threshold and chunk length are not learned from this right-hand side: they size the
// fermion-force solves.
int eo_propagator(Ctx &c, const double *phi, double2 *out, SolveStats *st) {
    const unsigned nbV = (unsigned)((c.V + kNT - 1) / kNT);
    hipLaunchKernelGGL(k_g5, dim3(nbV), dim3(kNT), 0, c.stream, c.V, c.eta);
    const int pred = c.eoPredIters, last = c.lastIters;
    const double scale = c.eoStopScale;
    if (onchip_eo(c)) {
        const int rc = onchip_eo_propagator(c, phi, out);
        return rc ? rc : read_stats(c, 1, st);
    }
    int rc = eo_solve(c, phi, 1, false, 0, 0, st);
    c.eoPredIters = pred;
    c.lastIters = last;
    c.eoStopScale = scale;
    if (rc) return rc;
    const EoArgs A = eo_args(c, 0, 0);
    hipLaunchKernelGGL(k_eo_propagator, dim3(nbV), dim3(kNT), 0, c.stream, A, phi, (const double2 *)c.x,
                       (const double2 *)c.eta, out);
    YCN_HIP(hipGetLastError());
    return YCN_OK;
}

int eo_drift(Ctx &c, const double *phi, double *drift, const StepCtl *ctl) {
    EoArgs A = eo_args(c, 0, 0);
    if (ctl) A.halt = &ctl->halt;
    const double fac = -c.p.g * (c.p.driftMode == 1 ? c.p.cutFraction * c.p.cutFraction : 1.0);
    hipLaunchKernelGGL(k_eo_drift, dim3((c.V + kNT - 1) / kNT, c.nRep), dim3(kNT), 0, c.stream, A, phi,
                       (const double2 *)c.x, (const double2 *)c.eta, drift, fac);
    YCN_HIP(hipGetLastError());
    return YCN_OK;
}

// ---------------------------------------------------------------------------
// Langevin steps without a host wait
// ---------------------------------------------------------------------------
// A step is k_step_begin, the coloured noise, the solve -- its setup, a fixed chunk schedule
// of the pipelined FP32 iteration with its reliable updates, k_step_check -- the drift and
// the update, all enqueued.  The solve and the drift may also be a captured graph
// (c.stepCapture), but a replay leaves longer gaps between its kernels than a stream does:
// sixteen steps at 1024 x 1024 38.4 ms replayed and 36.9 enqueued, 512 x 512 near the chiral
// point 19.1 and 17.9, 256 x 256 5.43 and 5.14, 128 x 96 11.28 and 11.20; enqueueing keeps
// the host busy instead (about 100 launches per step).  The schedule repeats the previous solve's rounds (eo_schedule), then `tail`
// chunks of 8.  A solve that needs more than the schedule holds halts the run
// (k_step_check): the later steps' kernels return at once except their chunk schedules,
// which keep iterating the halted solve (its FP32 and FP64 fields stay in c.phis and
// c.phiSolve), and the host finishes the halted step when it reads the control block at
// the end of the segment, then resumes.  Every chunk past the solve's end costs its
// launches (their kernels exit at once) and a halted step the rest of its segment, so the
// tail starts at one chunk, grows by one after each halted step and shrinks by one after
// four segments without one.  The field ping-pongs between the context's two buffers with
// a fixed step size and is updated in place with an adaptive one, so each schedule has at
// most two executables (one per field buffer).
constexpr int kStepSegment = 16;   // steps between two reads of the control block
constexpr int kMaxTail = 8;
constexpr size_t kMaxStepGraphs = 48;

bool eo_graph_eligible(const Ctx &c) {
    return c.stepGraphsOn && c.useGraphs && c.profTarget == PK_NONE && c.p.evenOdd && eo_available(c) &&
           eo_mixed(c) && c.p.precond == YCN_PRECOND_NONE && c.eoPredIters > 0;
}

// chunks of the schedule's main part for a predicted count when no earlier solve's
// reliable updates are known: the chunks the eager loop launches up to its first poll
static std::vector<int> eo_main_chunks(const Ctx &c, int pred) {
    const int every = std::max(1, c.p.reliableEvery);
    const int cap = c.p.cgMaxIter + every + (every & 1) + 8;
    std::vector<int> v;
    int itDone = 0;
    do {
        v.push_back(pf_chunk_len(c, pred, itDone));
        itDone += v.back();
    } while (itDone + pf_poll_margin(pred) < pred && itDone < cap);
    return v;
}

// The chunk schedule of a step: one chunk per reliable update of the previous
// solve (its longest system), each as long as that solve's round (the iterations between
// two reliable updates: up to a pause for the residual drop, to the stop, or to the end of
// an eager chunk) plus 2, rounded up to a multiple of 4, then `tail` chunks of 8.  The last
// schedule stays while it covers that with at most 7 launches to spare per round, so that
// consecutive solves mostly share one and its captured graphs.  (A launch after the systems have
// paused costs about 2 us: of the 56 of a 256 x 256 step with multiples of 8, 18 did.)  A
// round of this solve that ends a little later than the previous one's ends at the chunk
// boundary instead and the rest moves to the next round; a solve that needs more than
// the schedule holds halts the run.
constexpr int kTailRound = 8;
static std::vector<int> eo_schedule(Ctx &c, int tail) {
    std::vector<int> v;
    if (c.eoRounds.empty()) {
        v = eo_main_chunks(c, c.eoPredIters);
    } else {
        int prev = 0, total = 0;
        bool keep = c.eoRoundChunks.size() == c.eoRounds.size();
        for (int r : c.eoRounds) {
            const int need = std::max(4, r - prev + 2);
            if (keep) keep = need <= c.eoRoundChunks[v.size()] && c.eoRoundChunks[v.size()] <= need + 7;
            v.push_back((need + 3) / 4 * 4);
            prev = r;
        }
        if (keep) v = c.eoRoundChunks;
        c.eoRoundChunks = v;
        for (int n : v) total += n;
        // a solve with more reliable updates than CgState records ends after its last
        // recorded round: chunks of the reliable-update interval up to its iteration count
        if (prev < c.eoPredIters) {
            const int every = std::max(1, c.p.reliableEvery), nIt = every + (every & 1);
            const int want = std::min(c.eoPredIters, c.p.cgMaxIter) + 2;
            while (total < want) {
                v.push_back(nIt);
                total += nIt;
            }
        }
    }
    for (int k = 0; k < tail; ++k) v.push_back(kTailRound);
    return v;
}

// a step's solve and drift: the setup, the chunk schedule, k_step_check and the drift (the step's
// noise and update are launched around it by eo_enqueue_step)
static int eo_step_body(Ctx &c, int parity, const std::vector<int> &chunks) {
    const double *phiIn = c.phi[parity];
    const int nsys = c.nSys;
    int rc = eo_setup(c, phiIn, nsys, true, 1u, 0, true, c.ctl_d);
    for (int n : chunks)
        if (!rc) rc = eo_mixed_chunk(c, c.phiSolve, nsys, n, true);
    if (!rc) {
        hipLaunchKernelGGL(k_step_check, dim3(1), dim3(kWave), 0, c.stream, c.ctl_d, (const CgState *)c.cg_d, nsys,
                           c.p.cgTolMode == YCN_TOL_REL_TRUE ? 1 : 0);
        rc = eo_drift(c, phiIn, c.drift, c.ctl_d);   // fDrift.getForce(drift)
    }
    return rc;
}
static int eo_capture_step(Ctx &c, int parity, const std::vector<int> &chunks, hipGraphExec_t *out) {
    hipGraph_t g = nullptr;
    YCN_HIP(hipStreamBeginCapture(c.stream, hipStreamCaptureModeThreadLocal));
    int rc = eo_step_body(c, parity, chunks);
    const hipError_t le = hipGetLastError();
    const hipError_t ee = hipStreamEndCapture(c.stream, &g);
    if (rc || le != hipSuccess || ee != hipSuccess) {
        if (g) (void)hipGraphDestroy(g);
        if (!rc) {
            c.err = std::string("step capture: ") + hipGetErrorString(le != hipSuccess ? le : ee);
            rc = YCN_ERR_HIP;
        }
        return rc;
    }
    const hipError_t ie = hipGraphInstantiate(out, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (ie != hipSuccess) {
        c.err = std::string("step graph instantiation: ") + hipGetErrorString(ie);
        return YCN_ERR_HIP;
    }
    return YCN_OK;
}

// the executable of a schedule and field parity, captured at first use (the cache keeps
// the most recently used last); called only when no step graph is in flight: a segment
// fetches both of its executables before it launches a step
static int eo_step_graph(Ctx &c, int parity, const std::vector<int> &chunks, hipGraphExec_t *out) {
    for (size_t i = 0; i < c.stepGraphs.size(); ++i) {
        const Ctx::StepGraph e = c.stepGraphs[i];
        if (e.chunks == chunks && e.parity == parity) {
            c.stepGraphs.erase(c.stepGraphs.begin() + (long)i);
            c.stepGraphs.push_back(e);
            *out = e.exec;
            return YCN_OK;
        }
    }
    if (c.stepGraphs.size() >= kMaxStepGraphs) {
        (void)hipGraphExecDestroy(c.stepGraphs.front().exec);
        c.stepGraphs.erase(c.stepGraphs.begin());
    }
    const int rc = eo_capture_step(c, parity, chunks, out);
    if (rc) return rc;
    c.stepGraphs.push_back({chunks, parity, *out});
    return YCN_OK;
}

// While a segment runs on the GPU the host would only wait: it captures the schedules
// the next segment most likely needs, the current one with one chunk 4 launches shorter
// or longer (the rounds of consecutive solves move by a few iterations), for both field
// buffers, at most kPrecapture new ones per segment.  They go in at the cache's old end,
// so that they are evicted before anything the running segment uses.
constexpr int kPrecapture = 8;
static int eo_precapture(Ctx &c, const std::vector<int> &chunks, int nTail, bool bothParities) {
    int made = 0;
    const size_t nMain = chunks.size() - (size_t)nTail;
    for (size_t i = 0; i < nMain && made < kPrecapture; ++i)
        for (int d : {-4, 4}) {
            if (chunks[i] + d < 4) continue;
            std::vector<int> v = chunks;
            v[i] += d;
            for (int par = 0; par < (bothParities ? 2 : 1) && made < kPrecapture; ++par) {
                const int parity = bothParities ? par : c.cur;
                bool have = false;
                for (const Ctx::StepGraph &e : c.stepGraphs)
                    if (e.chunks == v && e.parity == parity) have = true;
                if (have) continue;
                if (c.stepGraphs.size() + 1 >= kMaxStepGraphs) return YCN_OK;   // never evict here
                hipGraphExec_t ex;
                const int rc = eo_capture_step(c, parity, v, &ex);
                if (rc) return rc;
                c.stepGraphs.insert(c.stepGraphs.begin(), {v, parity, ex});
                ++made;
            }
        }
    return YCN_OK;
}

// One step on the context stream, no host wait: k_step_begin, the coloured
// noise (on the noise stream beside the solve when the context has it, as a single step
// does: a graph with a second branch measured slower), the solve and drift (a captured graph where ex is given), then
// the update once the noise is there.  The noise reads the copy of the halt flag and
// counter k_step_begin made, so the solve's check kernel cannot change them under it.
static int eo_enqueue_step(Ctx &c, int parity, hipGraphExec_t ex, const std::vector<int> &chunks) {
    const bool fixed = c.p.adaptive == 0;
    double *phiIn = c.phi[parity], *phiOut = fixed ? c.phi[parity ^ 1] : c.phi[parity];
    StepCtl *ctlNoise = c.ctl_d + 1;
    const bool side = c.noiseSide && c.noiseStream;
    hipLaunchKernelGGL(k_step_begin, dim3(1), dim3(kWave), 0, c.stream, (const StepCtl *)c.ctl_d, ctlNoise, c.active,
                       c.nSys);
    int rc;
    if (side) {
        YCN_HIP(hipEventRecord(c.evMain, c.stream));
        YCN_HIP(hipStreamWaitEvent(c.noiseStream, c.evMain, 0));
        rc = noise_generate_ctl(c, c.noiseStream, ctlNoise, c.noise);   // cn()
        if (rc) return rc;
        YCN_HIP(hipEventRecord(c.evNoise, c.noiseStream));
    } else {
        rc = noise_generate_ctl(c, c.stream, ctlNoise, c.noise);   // cn()
        if (rc) return rc;
    }
    if (ex)
        YCN_HIP(hipGraphLaunch(ex, c.stream));   // fDrift.getForce(drift)
    else if ((rc = eo_step_body(c, parity, chunks)))
        return rc;
    if (side) YCN_HIP(hipStreamWaitEvent(c.stream, c.evNoise, 0));
    return bosonic_update_gated(c, fixed ? 1 : 0, phiIn, phiOut, &c.ctl_d->halt);   // kli.Run(kAll)
}

static void add_step_stats(SolveStats *tot, const SolveStats &st) {
    tot->iters_max += st.iters_max;
    tot->restarts += st.restarts;
    tot->converged &= st.converged;
    tot->rr_max = std::max(tot->rr_max, st.rr_max);
    tot->true_rel_max = std::max(tot->true_rel_max, st.true_rel_max);
    tot->iters_mean += st.iters_mean;
}

int eo_graph_run(Ctx &c, uint64_t step0, int nsteps, SolveStats *tot) {
    if (!c.ctl_d) {
        YCN_HIP(hipMalloc(&c.ctl_d, 2 * sizeof(StepCtl)));   // the control block and the noise's copy
        YCN_HIP(hipHostMalloc((void **)&c.ctl_h, sizeof(StepCtl), hipHostMallocDefault));
        YCN_HIP(hipMalloc(&c.phiSolve, sizeof(double) * (size_t)c.nRep * c.V));
    }
    const bool fixed = c.p.adaptive == 0;
    const int nsys = c.nSys;
    StepCtl &h = *c.ctl_h;
    h = StepCtl{};
    h.converged = 1;
    h.step = step0;
    h.stopScale = c.eoStopScale;
    h.lastIters = c.eoPredIters;
    h.nRounds = std::min((int)c.eoRounds.size(), kMaxRounds);
    for (int i = 0; i < h.nRounds; ++i) h.rounds[i] = c.eoRounds[i];
    YCN_HIP(hipMemcpyAsync(c.ctl_d, c.ctl_h, sizeof(StepCtl), hipMemcpyHostToDevice, c.stream));
    SolveStats host;   // figures of the steps the host finished
    int done = 0, rc;
    while (done < nsteps) {
        const int seg = std::min(kStepSegment, nsteps - done);
        const std::vector<int> chunks = eo_schedule(c, c.stepTail);
        const int p0 = c.cur;
        hipGraphExec_t ex[2] = {nullptr, nullptr};
        if (c.stepCapture && (rc = eo_step_graph(c, p0, chunks, &ex[p0]))) return rc;
        if (c.stepCapture && fixed && seg > 1 && (rc = eo_step_graph(c, p0 ^ 1, chunks, &ex[p0 ^ 1]))) return rc;
        for (int i = 0; i < seg; ++i) {
            const int parity = fixed ? p0 ^ (i & 1) : p0;
            if ((rc = eo_enqueue_step(c, parity, ex[parity], chunks))) return rc;
        }
        YCN_HIP(hipMemcpyAsync(c.ctl_h, c.ctl_d, sizeof(StepCtl), hipMemcpyDeviceToHost, c.stream));
        if (c.stepCapture && (rc = eo_precapture(c, chunks, c.stepTail, fixed))) return rc;
        if ((rc = spin_sync(c))) return rc;
        if (!h.halt) {
            c.cur = fixed ? p0 ^ (seg & 1) : p0;
            done += seg;
            if (++c.stepClean >= 4 && c.stepTail > 1) {
                --c.stepTail;
                c.stepClean = 0;
            }
        } else {
            // the halted step's solve is still in the context's state (the later steps'
            // chunk kernels may have iterated it further): finish it, then its drift and
            // update, eagerly; the field it started from is the one that step read
            const uint64_t first = step0 + (uint64_t)done;
            if (h.haltStep < first || h.haltStep >= first + (uint64_t)seg) {
                c.err = "enqueued steps: the control block names a step outside the segment";
                return YCN_ERR_HIP;
            }
            const int k = (int)(h.haltStep - first);
            c.cur = fixed ? p0 ^ (k & 1) : p0;
            SolveStats st;
            if ((rc = eo_mixed_loop(c, c.phi[c.cur], nsys, c.eoPredIters, &st))) return rc;
            if ((rc = eo_drift(c, c.phi[c.cur], c.drift))) return rc;
            if ((rc = bosonic_update(c, fixed ? 1 : 0))) return rc;
            add_step_stats(&host, st);
            ++c.haltedSteps;
            c.stepTail = std::min(c.stepTail + 1, kMaxTail);
            c.stepClean = 0;
            h.halt = 0;
            h.step = h.haltStep + 1;
            h.stopScale = c.eoStopScale;
            h.lastIters = st.iters_max;
            h.nRounds = (int)c.eoRounds.size();
            for (int i = 0; i < h.nRounds; ++i) h.rounds[i] = c.eoRounds[i];
            YCN_HIP(hipMemcpyAsync(c.ctl_d, c.ctl_h, sizeof(StepCtl), hipMemcpyHostToDevice, c.stream));
            done += k + 1;
        }
        // the next segment's schedule from the last finished step
        if (h.lastIters > 0) {
            c.eoPredIters = h.lastIters;
            c.eoRounds.assign(h.rounds, h.rounds + std::min(h.nRounds, kMaxRounds));
        }
        c.eoStopScale = h.stopScale;
    }
    c.lastIters = std::max(kGraphIters, c.eoPredIters);
    // the enqueued steps' figures (the last read of the block holds them all)
    SolveStats dev;
    dev.iters_max = (int)h.itersMaxSum;
    dev.iters_mean = h.itersMeanSum;
    dev.restarts = h.restarts;
    dev.converged = h.converged;
    dev.rr_max = h.rrMax;
    dev.true_rel_max = h.trueRelMax;
    add_step_stats(tot, dev);
    add_step_stats(tot, host);
    return YCN_OK;
}

}  // namespace ycn
