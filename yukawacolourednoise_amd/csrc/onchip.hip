// onchip.hip -- fermion-force solves that one workgroup holds on its CU.
//
// A lattice of a few thousand sites is far too small to fill the GPU, and a CG iteration
// of several launches spends its time in launch and reduction latency (16 x 16: four
// launches, 12.8 us per iteration; its arithmetic takes well under 1 us).  Here one
// workgroup per system runs the whole solve in one launch: noise vector, CG, true
// residual, restarts and the drift.  r, x, p live in registers (a thread owns one or two
// sites for the whole solve), p and D p pass through LDS, sums go through DPP and one LDS
// round, and nothing but eta touches memory until the end.  Vectors are packed real
// spinors (ycn_device.hpp).
//
// What bounds an iteration is LDS traffic and the chain of three barriers (p; D p with the
// first sum; the second sum): at 32 x 32 about 256 KB of LDS reads and writes per iteration,
// 2 000 cycles at 128 B per cycle.  Langevin steps in FP64, launched iterations against this with the step around it: 16 x 16
// 950 -> 107 us, 7 x 32 (no tile divides it) 1 060 -> 102 us, 32 x 32 1 250 -> 186 us.
#include <algorithm>
#include <cstdlib>

#include "bosonic.hpp"
#include "cg_fused.hpp"
#include "onchip.hpp"

namespace ycn {

// sites of a plain FP64 system one workgroup takes: p and D p are 64 B per site of LDS
// (128 KiB of the CU's 160), and two sites' vectors fill a thread's registers
constexpr int kOnchipSites = 2048;
constexpr int kOnchipThreads = 1024;

struct OnchipArgs {
    int Nt, Nx, V, nNoise;
    double r, M, g;
    double tol;
    int mode, maxIter, maxRestarts;
    double fac;          // drift factor
};

// A site's four neighbours, two registers: their sites (below kOnchipSites) in 15 bits
// each, (t+1, t-1) and (x+1, x-1), and the antiperiodic signs of the time hops in the two
// top bits of the first.  Unpacked they would take eight registers per site.
struct OnchipNbr {
    unsigned t, x;
};
__device__ __forceinline__ OnchipNbr onchip_nbr(const Nbr &n) {
    return {(unsigned)n.tf | (unsigned)n.tb << 15 | (n.sf < 0.0 ? 1u << 31 : 0u) | (n.sb < 0.0 ? 1u << 30 : 0u),
            (unsigned)n.xf | (unsigned)n.xb << 15};
}
__device__ __forceinline__ double onchip_sign(unsigned top) {   // +-1 by bit 31
    return __hiloint2double((int)(0x3FF00000u | (top & 0x80000000u)), 0);
}

// D (DAG = false) or D^dag applied at one site: own values a0, a1, neighbours from the
// planes B (plane stride V)
template <bool DAG, bool WR1>
__device__ __forceinline__ void onchip_dirac(const OnchipArgs &A, const double2 *B, OnchipNbr n, double d, double2 a0,
                                             double2 a1, double2 &o0, double2 &o1) {
    const double2 *B1 = B + A.V;
    n = {fresh(n.t), fresh(n.x)};
    const unsigned tf = n.t & 0x7FFF, tb = (n.t >> 15) & 0x7FFF, xf = n.x & 0x7FFF, xb = n.x >> 15;
    const double sf = onchip_sign(n.t), sb = onchip_sign(n.t << 1);
    if constexpr (WR1) {
        hop_flavour_r1<DAG, double, double2>(B[tf], B1[tf], sf, B[tb], B1[tb], sb, B[xf], B1[xf], B[xb], B1[xb], o0,
                                             o1);
    } else {
        hop_flavour_r<DAG, double, double2>(0.5 * (A.r + 1.0), 0.5 * (A.r - 1.0), 0.5 * A.r, 0.5, B[tf], B1[tf], sf,
                                            B[tb], B1[tb], sb, B[xf], B1[xf], B[xb], B1[xb], o0, o1);
    }
    o0 = make_double2(d * a0.x + o0.x, d * a0.y + o0.y);
    o1 = make_double2(d * a1.x + o1.x, d * a1.y + o1.y);
}

// The CG of k_cg_normal_fused / k_cg_c / k_fin_* (same recurrence, stopping and restart
// rules), whole.  DAG1: A = D D^dag, else D^dag D.  GEN: eta from the Philox streams (and
// written to eta), else read from it.  At the end w = D1 x of the last true residual is at
// hand: with DAG1 = false it is chi = D y, whose product with eta is the drift (nNoise = 1:
// drift; else the system's share, averaged by k_onchip_mean); with DAG1 = true it is
// D^dag x, written to wout (packed) for the measurement's propagator.
template <int K, bool WR1, bool DAG1, bool GEN>
__global__ void __launch_bounds__(kOnchipThreads)
k_onchip_plain(OnchipArgs A, const double *__restrict__ phi, const uint64_t *__restrict__ seeds, uint32_t streamBase,
               uint64_t step, double2 *__restrict__ eta, double2 *__restrict__ wout, double *__restrict__ drift,
               CgState *__restrict__ st) {
    extern __shared__ double2 sh[];
    __shared__ double red[2][16];
    const int sys = blockIdx.x, V = A.V, NT = blockDim.x;
    double2 *P = sh, *Q = sh + 2 * V;   // p and D1 p: two planes each
    eta += (size_t)sys * 2 * V;
    const double *ph = phi + (size_t)(sys / A.nNoise) * V;
    int turn = 0;

    OnchipNbr nb[K];
    double d[K];
    double2 x0[K], x1[K], r0[K], r1[K], p0[K], p1[K];
    double acc = 0.0;
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int s = threadIdx.x + k * NT;
        x0[k] = x1[k] = r0[k] = r1[k] = p0[k] = p1[k] = make_double2(0.0, 0.0);
        if (s < V) {
            const int t = s / A.Nx, x = s - t * A.Nx;
            nb[k] = onchip_nbr(neighbours(t, x, A.Nt, A.Nx));
            d[k] = 2.0 * A.r + A.M + A.g * ph[s];
            double2 b[2];
            if constexpr (GEN) {
                eta_planes<2>(seeds, streamBase, step, sys, A.nNoise, s, b);
                eta[s] = b[0];
                eta[V + s] = b[1];
            } else {
                b[0] = eta[s];
                b[1] = eta[V + s];
            }
            r0[k] = b[0];
            r1[k] = b[1];
            acc += b[0].x * b[0].x + b[0].y * b[0].y + b[1].x * b[1].x + b[1].y * b[1].y;
        }
    }
    double rr = onchip_sum(acc, red, turn);
    const double bn = sqrt(rr), stop = (A.mode == YCN_TOL_ABS_RECURSIVE) ? A.tol : A.tol * bn;
    bool run = 0 < A.maxIter && bn > stop;
    int iter = 0, restarts = 0, converged = run ? 0 : 1;
    double beta = 0.0, trueRel = 0.0;

    // w = D1 v through P and Q, leaving it in Q; o = D2 w; returns |w|^2, whose sum over the block
    // shares the barrier that publishes w
    auto normal_op = [&](const double2 *v0, const double2 *v1, double2 *w0, double2 *w1, double2 *o0, double2 *o1) {
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int s = threadIdx.x + k * NT;
            if (s < V) {
                P[s] = v0[k];
                P[V + s] = v1[k];
            }
        }
        __syncthreads();
        double ww = 0.0;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int s = threadIdx.x + k * NT;
            if (s < V) {
                onchip_dirac<DAG1, WR1>(A, P, nb[k], d[k], v0[k], v1[k], w0[k], w1[k]);
                Q[s] = w0[k];
                Q[V + s] = w1[k];
                ww += (w0[k].x * w0[k].x + w0[k].y * w0[k].y) + (w1[k].x * w1[k].x + w1[k].y * w1[k].y);
            }
        }
        ww = onchip_sum(ww, red, turn);
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int s = threadIdx.x + k * NT;
            o0[k] = o1[k] = make_double2(0.0, 0.0);
            if (s < V) onchip_dirac<!DAG1, WR1>(A, Q, nb[k], d[k], w0[k], w1[k], o0[k], o1[k]);
        }
        return ww;
    };

    double2 w0[K], w1[K], a0[K], a1[K];
    for (;;) {
        while (run) {
            const double inv = 1.0 / rr;   // ahead of the sum that beta waits for
#pragma unroll
            for (int k = 0; k < K; ++k) {
                p0[k] = make_double2(r0[k].x + beta * p0[k].x, r0[k].y + beta * p0[k].y);
                p1[k] = make_double2(r1[k].x + beta * p1[k].x, r1[k].y + beta * p1[k].y);
            }
            const double alpha = rr / normal_op(p0, p1, w0, w1, a0, a1);   // <p, A p> = |D1 p|^2
            double rn = 0.0;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                x0[k] = cadd(x0[k], cscl(alpha, p0[k]));
                x1[k] = cadd(x1[k], cscl(alpha, p1[k]));
                r0[k] = csub(r0[k], cscl(alpha, a0[k]));
                r1[k] = csub(r1[k], cscl(alpha, a1[k]));
                rn += (r0[k].x * r0[k].x + r0[k].y * r0[k].y) + (r1[k].x * r1[k].x + r1[k].y * r1[k].y);
            }
            rn = onchip_sum(rn, red, turn);
            beta = rn * inv;
            rr = rn;
            ++iter;
            if (iter >= A.maxIter || !(rn > stop * stop)) {
                run = false;
                converged = rn <= stop * stop ? 1 : 0;
            }
        }
        // true residual |b - A x| / |b|; in relative mode restart from it while above tol
        normal_op(x0, x1, w0, w1, a0, a1);
        double res = 0.0;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            const int s = threadIdx.x + k * NT;
            if (s < V) {
                const double2 e0 = csub(eta[s], a0[k]), e1 = csub(eta[V + s], a1[k]);
                a0[k] = e0;
                a1[k] = e1;
                res += (e0.x * e0.x + e0.y * e0.y) + (e1.x * e1.x + e1.y * e1.y);
            }
        }
        res = onchip_sum(res, red, turn);
        trueRel = bn > 0.0 ? sqrt(res) / bn : sqrt(res);
        if (A.mode != YCN_TOL_REL_TRUE) break;
        converged = trueRel <= A.tol ? 1 : 0;
        if (!(trueRel > A.tol && iter < A.maxIter && restarts < A.maxRestarts)) break;
        ++restarts;
        rr = res;
        beta = 0.0;
        run = true;
#pragma unroll
        for (int k = 0; k < K; ++k) {
            r0[k] = a0[k];
            r1[k] = a1[k];
        }
    }
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int s = threadIdx.x + k * NT;
        if (s >= V) continue;
        if constexpr (DAG1) {
            wout[s] = w0[k];
            wout[V + s] = w1[k];
        } else {
            const double2 e0 = eta[s], e1 = eta[V + s];
            const double sm = (w0[k].x * e0.x + w0[k].y * e0.y) + (w1[k].x * e1.x + w1[k].y * e1.y);
            drift[(size_t)sys * V + s] = A.nNoise == 1 ? A.fac * sm : sm;
        }
    }
    if (threadIdx.x == 0) {
        CgState &S = st[sys];
        S.iter = iter;
        S.restarts = restarts;
        S.converged = converged;
        S.rr = rr;
        S.true_rel = trueRel;
    }
}

// drift = fac times the mean of the noise vectors' shares
__global__ void __launch_bounds__(256)
k_onchip_mean(const double *__restrict__ share, double *__restrict__ drift, int V, int nNoise, double fac) {
    const int s = blockIdx.x * 256 + threadIdx.x;
    if (s >= V) return;
    const int rep = blockIdx.y;
    double acc = 0.0;
    for (int j = 0; j < nNoise; ++j) acc += share[((size_t)rep * nNoise + j) * V + s];
    drift[(size_t)rep * V + s] = fac * acc / (double)nNoise;
}

// The plain solvers' packed solves on lattices of up to kOnchipSites, unless a tile is
// forced through the environment or a kernel of the launched iterations is being timed.
// A lattice larger than that takes launches.
bool onchip_plain(const Ctx &c) {
    return c.onchip && c.V <= kOnchipSites && c.p.precond == YCN_PRECOND_NONE && c.profTarget == PK_NONE;
}

int onchip_init(Ctx &c) {
    c.onchip = true;
    for (const char *e : {"YCN_TILE", "YCN_TILE32", "YCN_TILE_EO", "YCN_TILE_EO32", "YCN_EO_FIN"})
        if (std::getenv(e)) c.onchip = false;
    if (const char *e = std::getenv("YCN_ONCHIP")) c.onchip = c.onchip && std::atoi(e) != 0;
    return YCN_OK;
}

template <int K, bool DAG1, bool GEN>
static int launch_plain(Ctx &c, const OnchipArgs &A, int nsys, int threads, const double *phi, uint32_t streamBase,
                        uint64_t step, double2 *wout, double *drift) {
    auto *k = A.r == 1.0 ? &k_onchip_plain<K, true, DAG1, GEN> : &k_onchip_plain<K, false, DAG1, GEN>;
    const size_t lds = sizeof(double2) * 4 * (size_t)A.V;
    hipLaunchKernelGGL(k, dim3(nsys), dim3(threads), lds, c.stream, A, phi, (const uint64_t *)c.seed_d, streamBase,
                       step, c.eta, wout, drift, c.cg_d);
    YCN_HIP(hipGetLastError());
    return YCN_OK;
}

template <bool DAG1, bool GEN>
static int onchip_launch(Ctx &c, const double *phi, int nsys, uint32_t streamBase, uint64_t step, double2 *wout,
                         double *drift) {
    OnchipArgs A;
    A.Nt = c.p.Nt;
    A.Nx = c.p.Nx;
    A.V = c.V;
    A.nNoise = c.nNoise;
    A.r = c.p.r;
    A.M = c.p.M;
    A.g = c.p.g;
    A.tol = c.p.cgTol;
    A.mode = c.p.cgTolMode;
    A.maxIter = c.p.cgMaxIter;
    A.maxRestarts = 4;
    A.fac = -c.p.g * (c.p.driftMode == 1 ? c.p.cutFraction * c.p.cutFraction : 1.0);
    const int threads = std::min(kOnchipThreads, (c.V + kWave - 1) / kWave * kWave);
    return c.V <= kOnchipThreads ? launch_plain<1, DAG1, GEN>(c, A, nsys, threads, phi, streamBase, step, wout, drift)
                                 : launch_plain<2, DAG1, GEN>(c, A, nsys, threads, phi, streamBase, step, wout, drift);
}

// where a solve leaves its systems' drifts: the drift itself, or with several noise vectors
// their shares in scratch, which onchip_mean averages
double *onchip_share(Ctx &c) { return c.nNoise == 1 ? c.drift : reinterpret_cast<double *>(c.Ap); }

int onchip_mean(Ctx &c) {
    if (c.nNoise == 1) return YCN_OK;
    const double fac = -c.p.g * (c.p.driftMode == 1 ? c.p.cutFraction * c.p.cutFraction : 1.0);
    hipLaunchKernelGGL(k_onchip_mean, dim3((c.V + 255) / 256, c.nRep), dim3(256), 0, c.stream,
                       (const double *)onchip_share(c), c.drift, c.V, c.nNoise, fac);
    YCN_HIP(hipGetLastError());
    return YCN_OK;
}

// the fermion force of every system into c.drift; the states stay on the device
int onchip_force(Ctx &c, const double *phi, uint32_t streamBase, uint64_t step) {
    const int rc = onchip_launch<false, true>(c, phi, c.nSys, streamBase, step, nullptr, onchip_share(c));
    return rc ? rc : onchip_mean(c);
}

// D^-1 of the packed source in c.eta (system 0, c.nNoise = 1) into out
int onchip_propagator(Ctx &c, const double *phi, double2 *out) {
    return onchip_launch<true, false>(c, phi, 1, 0, 0, out, nullptr);
}

// ---------------------------------------------------------------------------
// Langevin steps whose solves are held on chip
// ---------------------------------------------------------------------------
// The bosonic drift, the adaptive step size and the Euler-Maruyama update of one replica by one
// block, up to four sites per thread (k_bosonic_max, k_fin_eps and k_evolve, or k_update_fixed,
// in one launch: same arithmetic), and the step's report to the host.  in == out where the step
// is adaptive: every neighbour is read before the barrier of the maximum, and written after it.
constexpr int kUpdateSites = 4;
__global__ void __launch_bounds__(kOnchipThreads)
k_onchip_update(const double *in, double *out, const double *__restrict__ drift, const double *__restrict__ noise,
                const double *__restrict__ m2, double lam6, int Nt, int Nx, double epsBar, int adaptive,
                StepState *__restrict__ ss, const CgState *__restrict__ st, int nNoise, StepReport *report,
                uint32_t seq) {
    __shared__ double red[2][16];
    const int rep = blockIdx.x, V = Nt * Nx;
    const size_t off = (size_t)rep * V;
    const double *ph = in + off;
    double f[kUpdateSites], d[kUpdateSites], mx = 0.0;
    int turn = 0;
#pragma unroll
    for (int k = 0; k < kUpdateSites; ++k) {
        const int s = threadIdx.x + k * kOnchipThreads;
        f[k] = d[k] = 0.0;
        if (s < V) {
            f[k] = ph[s];
            d[k] = drift[off + s] + bosonic_drift(ph, s, Nt, Nx, m2[rep], lam6);
            mx = fmax(mx, fabs(d[k]));
        }
    }
    double e = epsBar;
    int clamp = 0;
    if (adaptive) {
        mx = onchip_max(mx, red, turn);
        if (mx > 1e5) { mx = 1e5; clamp = 1; }
        else if (mx < 1e-5) { mx = 1e-5; clamp = 1; }
        e = epsBar * 30.0 / mx;
    }
    const double fact = sqrt(2.0 * e);
#pragma unroll
    for (int k = 0; k < kUpdateSites; ++k) {
        const int s = threadIdx.x + k * kOnchipThreads;
        if (s < V) out[off + s] = f[k] - (e * d[k] + fact * noise[off + s]);
    }
    if (threadIdx.x) return;
    StepState &S = ss[rep];
    S.eps = e;
    S.tL += e;
    if (adaptive) {
        S.maxDrift = mx;
        S.clamps += clamp;
    }
    StepReport R{};
    R.eps = e;
    R.converged = 1;
    for (int j = 0; j < nNoise; ++j) {
        const CgState &g = st[rep * nNoise + j];
        R.iterMax = max(R.iterMax, g.iter);
        R.iterSum += g.iter;
        R.restarts = max(R.restarts, g.restarts);
        R.converged &= g.converged;
        R.rrMax = fmax(R.rrMax, g.rr);
        R.trueRelMax = fmax(R.trueRelMax, g.true_rel);
        if (g.need > 0.0 && g.stop0 > 0.0) R.ratio = fmax(R.ratio, g.need / g.stop0);
    }
    StepReport *to = report + rep;
    to->eps = R.eps;
    to->iterSum = R.iterSum;
    to->rrMax = R.rrMax;
    to->trueRelMax = R.trueRelMax;
    to->ratio = R.ratio;
    to->iterMax = R.iterMax;
    to->restarts = R.restarts;
    to->converged = R.converged;
    __hip_atomic_store(&to->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Measured at this form (one launch each for noise, force and update, reports in pinned memory,
// one host wait for up to kRunSlots steps) against three to five launches, a side stream, two
// copies and two or three waits per step: 16 x 16 adaptive, step by step, 170 -> 100 us; 32 x 32
// 211 -> 187 us; 64 chains of 64 x 64 444 -> 397 us.
bool onchip_steps(const Ctx &c) {
    return (onchip_eo(c) || (!c.p.evenOdd && onchip_plain(c))) && c.V <= kUpdateSites * kOnchipThreads;
}

constexpr int kRunSlots = 64;   // steps in flight before the host waits for their reports
// Steps whose noise one launch makes: a field takes one block 10 to 20 us (16 x 16 to 64 x 64), as
// long as a whole launch of them does while the chip has compute units left, so a run of 16 steps
// pays for one (32 x 32: 14 us of a 198 us step before).
constexpr int kNoiseSteps = 16;

static int run_init(Ctx &c) {
    if (!c.report) {
        YCN_HIP(hipHostMalloc((void **)&c.report, sizeof(StepReport) * kRunSlots * c.nRep, hipHostMallocDefault));
        for (int i = 0; i < kRunSlots * c.nRep; ++i) c.report[i].seq = 0;
    }
    // noise of several steps ahead, in at most 64 MiB
    if (!c.noiseRun) {
        const size_t one = (size_t)c.nRep * c.V, fit = ((size_t)64 << 20) / (sizeof(double) * one);
        c.noiseSteps = (int)std::max<size_t>(1, std::min<size_t>(kNoiseSteps, fit));
        YCN_HIP(hipMalloc(&c.noiseRun, sizeof(double) * one * c.noiseSteps));
    }
    if (c.p.evenOdd && !c.ratio) YCN_HIP(hipMalloc(&c.ratio, sizeof(double) * 2 * ((size_t)c.nSys + 1)));
    return YCN_OK;
}

void onchip_free(Ctx &c) {
    if (c.report) (void)hipHostFree(c.report);
    if (c.ratio) (void)hipFree(c.ratio);
    if (c.noiseRun) (void)hipFree(c.noiseRun);
    c.noiseRun = nullptr;
    c.report = nullptr;
    c.ratio = nullptr;
}

// wait until a step's reports of every replica carry its number; an error or an idle stream
// without them ends the wait
static int wait_report(Ctx &c, const StepReport *r, uint32_t seq) {
    ++c.hostSyncs;
    bool idle = false;
    for (int rep = 0; rep < c.nRep; ++rep)
        for (int spin = 0; __atomic_load_n(&r[rep].seq, __ATOMIC_ACQUIRE) != seq; ++spin) {
            if (idle) {
                c.err = "a Langevin step ended without its report";
                return YCN_ERR_HIP;
            }
            if ((spin & 1023) != 1023) continue;
            const hipError_t e = hipStreamQuery(c.stream);
            if (e == hipSuccess)
                idle = __atomic_load_n(&r[rep].seq, __ATOMIC_ACQUIRE) != seq;
            else if (e != hipErrorNotReady)
                YCN_HIP(e);
        }
    return YCN_OK;
}

int onchip_run(Ctx &c, uint64_t step0, int nsteps, SolveStats *tot, double *eps) {
    int rc = run_init(c);
    const bool fixed = c.p.adaptive == 0;
    for (int done = 0; done < nsteps && !rc;) {
        const int seg = std::min(kRunSlots, nsteps - done);
        const uint32_t first = c.reportSeq + 1;
        for (int i = 0; i < seg; ++i) {
            const uint64_t step = step0 + (uint64_t)(done + i);
            double *in = c.phi[c.cur], *out = fixed ? c.phi[c.cur ^ 1] : in;
            const int ahead = i % c.noiseSteps;
            if (ahead == 0 && (rc = noise_generate_steps(c, step, std::min(seg - i, c.noiseSteps), c.noiseRun)))
                return rc;                                                                          // cn()
            const double *noise = c.noiseRun + (size_t)ahead * c.nRep * c.V;
            rc = c.p.evenOdd ? onchip_eo_force(c, in, 1u, step, i > 0) : onchip_force(c, in, 1u, step);
            if (rc) return rc;                                                                      // getForce(drift)
            hipLaunchKernelGGL(k_onchip_update, dim3(c.nRep), dim3(kOnchipThreads), 0, c.stream, (const double *)in, out,
                               (const double *)c.drift, noise, (const double *)c.m2_d,
                               c.p.lambda / 6.0, c.p.Nt, c.p.Nx, c.epsBar, c.p.adaptive, c.step_d,
                               (const CgState *)c.cg_d, c.nNoise, c.report + (size_t)i * c.nRep, ++c.reportSeq);
            YCN_HIP(hipGetLastError());                                                             // kli.Run(kAll)
            if (fixed) c.cur ^= 1;
        }
        if ((rc = wait_report(c, c.report + (size_t)(seg - 1) * c.nRep, first + (uint32_t)(seg - 1)))) return rc;
        double ratio = 0.0;
        for (int i = 0; i < seg; ++i) {
            SolveStats st;
            double sum = 0.0;
            ratio = 0.0;
            for (int rep = 0; rep < c.nRep; ++rep) {
                const StepReport &r = c.report[(size_t)i * c.nRep + rep];
                st.iters_max = std::max(st.iters_max, r.iterMax);
                st.restarts = std::max(st.restarts, r.restarts);
                st.converged &= r.converged;
                st.rr_max = std::max(st.rr_max, r.rrMax);
                st.true_rel_max = std::max(st.true_rel_max, r.trueRelMax);
                sum += r.iterSum;
                if (eps && done + i == nsteps - 1) eps[rep] = r.eps;
                ratio = std::max(ratio, r.ratio);
            }
            tot->iters_max += st.iters_max;
            tot->restarts += st.restarts;
            tot->converged &= st.converged;
            tot->rr_max = std::max(tot->rr_max, st.rr_max);
            tot->true_rel_max = std::max(tot->true_rel_max, st.true_rel_max);
            tot->iters_mean += sum / c.nSys;
            // the threshold the next solve starts from, as the device derives it along the segment
            if (c.p.evenOdd && c.p.cgTolMode == YCN_TOL_REL_TRUE && ratio > 0.0)
                c.eoStopScale = std::min(1.0, std::max(1e-3, 0.9 * ratio));
        }
        done += seg;
    }
    return rc;
}

}  // namespace ycn
