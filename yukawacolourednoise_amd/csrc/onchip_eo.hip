// onchip_eo.hip -- even-odd preconditioned fermion-force solves that one workgroup holds on
// its CU: noise vector, right-hand side, CG on the Schur complement, true residual and the
// drift of one system in one launch (see evenodd.hip for the equations, onchip.hip for the
// plain solver's counterpart).
//
// A system's half-lattice vectors are small (64 x 64: 2048 even sites, 64 KB each), so a thread
// owns up to two sites of each parity for the whole solve: r, p, x and the diagonals in
// registers, one vector of each parity in LDS for the hops.  The two sites follow each other in
// time and the odd and the even site of an entry are x neighbours, so a hop takes its own
// entry's value and half of its time neighbours from registers.
//
// FP64 throughout, also where the context asks for mixed precision: held on chip a vector costs
// no bandwidth, and FP64 instructions issue at the rate of FP32 ones, so FP32 iterations would
// gain nothing and pay for reliable updates (64 x 64, 512 systems, four sites a thread: 519 us a
// solve in mixed precision, 455 in FP64).
//
// What bounds it: LDS and VALU issue about equally, in a chain of five barriers per iteration.
#include <algorithm>
#include <cmath>

#include "cg_fused.hpp"
#include "onchip.hpp"

namespace ycn {

constexpr int kOnchipEoThreads = 1024;
constexpr int kOnchipEoSites = 2 * kOnchipEoThreads;   // even sites of a system: two per thread

struct OnchipEoArgs {
    int Nt, Nx, Nh, V, Vh, nNoise;
    double r, M, g;
    double tol, stopScale, fac;
    int mode, maxIter, maxRestarts;
};

// both spins of a site, each (flavour 0, flavour 1)
struct Spin2 {
    double2 a, b;
};
__device__ __forceinline__ double sq(const Spin2 &v) {
    return (v.a.x * v.a.x + v.a.y * v.a.y) + (v.b.x * v.b.x + v.b.y * v.b.y);
}
__device__ __forceinline__ Spin2 scaled(double s, const Spin2 &v) { return {cscl(s, v.a), cscl(s, v.b)}; }
// u + s v
__device__ __forceinline__ Spin2 axpy(const Spin2 &u, double s, const Spin2 &v) {
    return {make_double2(u.a.x + s * v.a.x, u.a.y + s * v.a.y), make_double2(u.b.x + s * v.b.x, u.b.y + s * v.b.y)};
}

// LDS entries of 16 bytes, one per spin: [spin][i][thread], so that the lanes of every access
// lie side by side
template <int K>
struct EoLds {
    static constexpr int row = 16 * kOnchipEoThreads, plane = K * row, bytes = 2 * plane;
    static __device__ __forceinline__ double2 get(const char *B, unsigned a, int i, int spin) {
        return *reinterpret_cast<const double2 *>(B + a + i * row + spin * plane);
    }
    static __device__ __forceinline__ void put(char *B, unsigned a, int i, const Spin2 &v) {
        *reinterpret_cast<double2 *>(B + a + i * row) = v.a;
        *reinterpret_cast<double2 *>(B + a + i * row + plane) = v.b;
    }
};

// A thread's neighbours as LDS addresses of their threads: the strips after and before its own
// in time, and the columns before and after it; the antiperiodic signs of the time hops that
// leave the strip; and whether its first row is odd (K = 1; strips of two start on even rows).
struct EoNbr {
    unsigned tf, tb, xm, xp;
    unsigned sf, sb;   // sign bits
    bool odd;
};
__device__ __forceinline__ double2 flip(double2 v, unsigned sign) {
    const long long m = (long long)sign << 32;
    return make_double2(__longlong_as_double(__double_as_longlong(v.x) ^ m),
                        __longlong_as_double(__double_as_longlong(v.y) ^ m));
}

// K (DAG) or H onto the thread's sites of parity PAR, from the other parity's vector: `src` its
// own entries, B the LDS copy.  In x one neighbour is the own entry u and the other, w, lies
// behind the even sites of even rows and the odd sites of odd rows, else ahead: the hop's x
// terms are r/2 (u + w) and -+(u - w)/2.
template <bool DAG, int PAR, bool WR1, int K>
__device__ __forceinline__ void eo_hop_own(const OnchipEoArgs &A, const char *B, const EoNbr &n, const Spin2 (&src)[K],
                                           Spin2 (&o)[K]) {
    using L = EoLds<K>;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        const bool odd = K == 1 ? n.odd : (i & 1);
        const bool ahead = odd != (PAR == 1);
        const unsigned wa = ahead ? n.xp : n.xm;
        // the term (Xb - Xf) / 2 of H is s (u - w); K has the neighbours swapped
        const double s = (ahead != DAG) ? 0.5 : -0.5;
        const Spin2 u = src[i], w = {L::get(B, wa, i, 0), L::get(B, wa, i, 1)};
        // the neighbours ahead and behind in time, one spin of each (r = 1: projectors)
        auto fwd = [&](int spin) {
            if (i + 1 < K) return spin ? src[i + 1 < K ? i + 1 : i].b : src[i + 1 < K ? i + 1 : i].a;
            return flip(L::get(B, n.tf, 0, spin), n.sf);
        };
        auto bwd = [&](int spin) {
            if (i > 0) return spin ? src[i > 0 ? i - 1 : i].b : src[i > 0 ? i - 1 : i].a;
            return flip(L::get(B, n.tb, K - 1, spin), n.sb);
        };
        const double2 t0 = DAG ? fwd(0) : bwd(0), t1 = DAG ? bwd(1) : fwd(1);
        const double hp = WR1 ? 1.0 : 0.5 * (A.r + 1.0), hr = WR1 ? 0.5 : 0.5 * A.r;
        o[i].a.x = hp * t0.x + hr * (u.a.x + w.a.x) + s * (u.b.x - w.b.x);
        o[i].a.y = hp * t0.y + hr * (u.a.y + w.a.y) + s * (u.b.y - w.b.y);
        o[i].b.x = hp * t1.x + hr * (u.b.x + w.b.x) + s * (u.a.x - w.a.x);
        o[i].b.y = hp * t1.y + hr * (u.b.y + w.b.y) + s * (u.a.y - w.a.y);
        if constexpr (!WR1) {
            const double hm = 0.5 * (A.r - 1.0);
            const double2 m0 = DAG ? bwd(0) : fwd(0), m1 = DAG ? fwd(1) : bwd(1);
            o[i].a.x += hm * m0.x;
            o[i].a.y += hm * m0.y;
            o[i].b.x += hm * m1.x;
            o[i].b.y += hm * m1.y;
        }
        o[i] = {make_double2(-o[i].a.x, -o[i].a.y), make_double2(-o[i].b.x, -o[i].b.y)};
    }
}

// The stopping, tightening and restart rules are those of the launched FP64 solver (k_fin_beta,
// k_fin_eo_true).  GEN: eta from the Philox streams, written to eta; else read from it.  PROP:
// out = gamma_5 i chi on the full lattice (the measurement's propagator); else the system's
// drift (nNoise = 1) or its share of it.
template <int K, bool WR1, bool GEN, bool PROP>
__global__ void __launch_bounds__(kOnchipEoThreads)
k_onchip_eo(OnchipEoArgs A, const double *__restrict__ phi, const uint64_t *__restrict__ seeds, uint32_t streamBase,
            uint64_t step, double2 *eta, double2 *bg, double *__restrict__ drift, double2 *__restrict__ out,
            CgState *__restrict__ st, const double *__restrict__ ratioIn, double *__restrict__ ratioOut, int nsys) {
    using L = EoLds<K>;
    extern __shared__ double2 sh[];
    __shared__ double red[2][16];
    const int sys = blockIdx.x, V = A.V, Vh = A.Vh, Nh = A.Nh;
    char *const E = reinterpret_cast<char *>(sh), *const O = E + L::bytes;
    eta += (size_t)sys * 2 * V;
    bg += (size_t)sys * 2 * Vh;
    const double *ph = phi + (size_t)(sys / A.nNoise) * V;
    int turn = 0;

    // strip `strip` of K rows at column pair `col`: the even and odd sites (strip K + i, col)
    const int strips = A.Nt / K, strip = threadIdx.x / Nh, col = threadIdx.x - strip * Nh;
    const bool own = strip < strips;
    EoNbr n;
    {
        const int sf = strip + 1 == strips ? 0 : strip + 1, sb = strip == 0 ? strips - 1 : strip - 1;
        n.tf = 16 * (sf * Nh + col);
        n.tb = 16 * (sb * Nh + col);
        n.xm = 16 * (strip * Nh + (col == 0 ? Nh - 1 : col - 1));
        n.xp = 16 * (strip * Nh + (col == Nh - 1 ? 0 : col + 1));
        n.sf = strip + 1 == strips ? 0x80000000u : 0u;
        n.sb = strip == 0 ? 0x80000000u : 0u;
        n.odd = (strip * K) & 1;
        if (!own) n.tf = n.tb = n.xm = n.xp = 0;   // idle threads read entry 0, and no one reads theirs
    }
    const unsigned me = 16 * threadIdx.x;
    auto full = [&](int i, int par) {   // full-lattice site (formed anew: used before and after the iterations)
        const int th = (int)fresh(threadIdx.x), q = th / Nh, t = q * K + i;
        return t * A.Nx + 2 * (th - q * Nh) + ((t + par) & 1);
    };
    auto put = [&](char *B, const Spin2 (&v)[K]) {
#pragma unroll
        for (int i = 0; i < K; ++i) L::put(B, me, i, v[i]);
        __syncthreads();
    };
    const Spin2 zero = {make_double2(0.0, 0.0), make_double2(0.0, 0.0)};

    // ---- noise vector, b_e = eta_e - K_eo A_o^-1 eta_o, r = S^T b ----
    double de[K], io[K];   // d on the even sites, 1 / d on the odd ones (idle threads: zeros)
    Spin2 r[K], p[K], x[K], v[K], u[K];
    double acc = 0.0;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        r[i] = p[i] = x[i] = v[i] = u[i] = zero;
        de[i] = io[i] = 0.0;
    }
    if (own) {
#pragma unroll
        for (int i = 0; i < K; ++i) {
            de[i] = 2.0 * A.r + A.M + A.g * ph[full(i, 0)];
            io[i] = 1.0 / (2.0 * A.r + A.M + A.g * ph[full(i, 1)]);
        }
#pragma unroll 1
        for (int q = 0; q < 2 * K; ++q) {
            const int i = q >> 1, par = q & 1, f = full(i, par);
            double2 e[2];
            if constexpr (GEN) {
                eta_planes<2>(seeds, streamBase, step, sys, A.nNoise, f, e);
                eta[f] = e[0];
                eta[V + f] = e[1];
            } else {
                e[0] = eta[f];
                e[1] = eta[V + f];
            }
            const Spin2 w = {e[0], e[1]};
            acc += sq(w);
#pragma unroll
            for (int k = 0; k < K; ++k)
                if (k == i) {
                    if (par)
                        u[k] = scaled(io[k], w);   // A_o^-1 eta_o
                    else
                        v[k] = w;
                }
        }
    }
    put(O, u);
    eo_hop_own<true, 0, WR1, K>(A, O, n, u, p);
#pragma unroll
    for (int i = 0; i < K; ++i) {
        v[i] = axpy(v[i], -1.0, p[i]);
        if (!own) v[i] = zero;
        p[i] = zero;
        if (own) {
            bg[threadIdx.x + i * strips * Nh] = v[i].a;
            bg[Vh + threadIdx.x + i * strips * Nh] = v[i].b;
        }
    }
    put(E, v);
    eo_hop_own<false, 1, WR1, K>(A, E, n, v, u);
#pragma unroll
    for (int i = 0; i < K; ++i) u[i] = scaled(io[i], u[i]);
    put(O, u);
    eo_hop_own<false, 0, WR1, K>(A, O, n, u, r);
    double rn = 0.0;
#pragma unroll
    for (int i = 0; i < K; ++i) {
        r[i] = own ? axpy(scaled(de[i], v[i]), -1.0, r[i]) : zero;
        rn += sq(r[i]);
    }
    const double enorm2 = onchip_sum(acc, red, turn);
    double rr = onchip_sum(rn, red, turn);
    double beta = 0.0, need = 0.0, trueRel = 0.0;
    // the starting threshold: the context's, or learned from the solve before as
    // eo_learn_stop_scale does (ratioIn: that solve's ratios, and the scale it started from)
    double scale = A.stopScale;
    if (ratioIn) {
        double m = 0.0;
        for (int k = threadIdx.x; k < nsys; k += blockDim.x) m = fmax(m, ratioIn[k]);
        m = onchip_max(m, red, turn);
        scale = m > 0.0 ? fmin(1.0, fmax(1e-3, 0.9 * m)) : ratioIn[nsys];
    }
    const double stop0 = A.mode == YCN_TOL_ABS_RECURSIVE ? A.tol : A.tol * sqrt(rr);
    double stop = A.mode == YCN_TOL_REL_TRUE ? stop0 * scale : stop0;
    int iter = 0, restarts = 0;
    bool run = 0 < A.maxIter && sqrt(rr) > stop;
    int converged = run ? 0 : 1;

    for (;;) {
        while (run) {
            const double inv = 1.0 / rr;   // ahead of the sum that beta waits for
            // p = r + beta p; U = A_o^-1 K p; v = S p; W = A_o^-1 H v; Ap = S^T v.  O is written
            // and E read between the same barriers, and the other way round, so one barrier
            // separates each stage from the next.
#pragma unroll
            for (int i = 0; i < K; ++i) p[i] = axpy(r[i], beta, p[i]);
            put(E, p);
            eo_hop_own<true, 1, WR1, K>(A, E, n, p, u);
#pragma unroll
            for (int i = 0; i < K; ++i) u[i] = scaled(io[i], u[i]);
            put(O, u);
            eo_hop_own<true, 0, WR1, K>(A, O, n, u, v);
            double mu = 0.0;
#pragma unroll
            for (int i = 0; i < K; ++i) {
                v[i] = own ? axpy(scaled(de[i], p[i]), -1.0, v[i]) : zero;
                mu += sq(v[i]);
                L::put(E, me, i, v[i]);
            }
            mu = onchip_sum(mu, red, turn);   // its barrier publishes v
            eo_hop_own<false, 1, WR1, K>(A, E, n, v, u);
#pragma unroll
            for (int i = 0; i < K; ++i) u[i] = scaled(io[i], u[i]);
            put(O, u);
            const double alpha = rr / mu;
            Spin2 ap[K];
            eo_hop_own<false, 0, WR1, K>(A, O, n, u, ap);
            double rho = 0.0;
#pragma unroll
            for (int i = 0; i < K; ++i) {
                ap[i] = axpy(scaled(de[i], v[i]), -1.0, ap[i]);
                x[i] = axpy(x[i], alpha, p[i]);
                r[i] = own ? axpy(r[i], -alpha, ap[i]) : zero;
                rho += sq(r[i]);
            }
            rho = onchip_sum(rho, red, turn);
            ++iter;
            beta = rho * inv;
            rr = rho;
            if (iter >= A.maxIter || !(rho > stop * stop)) {
                run = false;
                converged = rho <= stop * stop ? 1 : 0;
            }
        }
        // true residual |b - S x| / |eta|; u = A_o^-1 K x is kept for the drift
        put(E, x);
        eo_hop_own<true, 1, WR1, K>(A, E, n, x, u);
#pragma unroll
        for (int i = 0; i < K; ++i) u[i] = scaled(io[i], u[i]);
        put(O, u);
        eo_hop_own<true, 0, WR1, K>(A, O, n, u, v);
        double res = 0.0;
#pragma unroll
        for (int i = 0; i < K; ++i)
            if (own) {
                const Spin2 b = {bg[threadIdx.x + i * strips * Nh], bg[Vh + threadIdx.x + i * strips * Nh]};
                res += sq(axpy(axpy(b, -de[i], x[i]), 1.0, v[i]));
            }
        res = onchip_sum(res, red, turn);
        trueRel = enorm2 > 0.0 ? sqrt(res / enorm2) : sqrt(res);
        if (A.mode != YCN_TOL_REL_TRUE) break;
        if (trueRel > 0.0) need = sqrt(rr) * A.tol / trueRel;
        converged = trueRel <= A.tol ? 1 : 0;
        if (!(trueRel > A.tol && iter < A.maxIter && restarts < A.maxRestarts)) break;
        ++restarts;   // go on from this state with the threshold lowered by what is missing
        stop = sqrt(rr) * 0.5 * A.tol / trueRel;
        run = true;
    }

    // chi_o = A_o^-1 (eta_o - K_oe chi_e), and the drift or the propagator
    if (own) {
#pragma unroll
        for (int i = 0; i < K; ++i)
#pragma unroll
            for (int par = 0; par < 2; ++par) {
                const int f = full(i, par);
                const Spin2 e = {eta[f], eta[V + f]};
                const Spin2 ch = par ? axpy(scaled(io[i], e), -1.0, u[i]) : x[i];
                if constexpr (PROP) {
                    out[f] = ch.b;
                    out[V + f] = make_double2(-ch.a.x, -ch.a.y);
                } else {
                    const double sm = (ch.a.x * e.a.x + ch.a.y * e.a.y) + (ch.b.x * e.b.x + ch.b.y * e.b.y);
                    drift[(size_t)sys * V + f] = A.nNoise == 1 ? A.fac * sm : sm;
                }
            }
    }
    if (threadIdx.x == 0) {
        CgState &s = st[sys];
        s.iter = iter;
        s.restarts = restarts;
        s.converged = converged;
        s.rr = rr;
        s.true_rel = trueRel;
        s.need = need;
        s.stop0 = stop0;
        if (ratioOut) {
            ratioOut[sys] = need > 0.0 && stop0 > 0.0 ? need / stop0 : 0.0;
            if (sys == 0) ratioOut[nsys] = scale;
        }
    }
}

// Even-odd solves of systems of up to kOnchipEoSites even sites, unless a tile is forced
// through the environment or a kernel of the launched iterations is being timed.
bool onchip_eo(const Ctx &c) {
    return c.onchip && c.p.evenOdd && eo_available(c) && c.V / 2 <= kOnchipEoSites && c.profTarget == PK_NONE;
}

// bg: scratch for b_e; no two of bg, drift and out may be the same memory
template <bool GEN, bool PROP>
static int launch_eo(Ctx &c, const double *phi, int nsys, uint32_t streamBase, uint64_t step, double2 *bg,
                     double *drift, double2 *out, const double *ratioIn, double *ratioOut) {
    OnchipEoArgs A;
    A.Nt = c.p.Nt;
    A.Nx = c.p.Nx;
    A.Nh = c.p.Nx / 2;
    A.V = c.V;
    A.Vh = c.V / 2;
    A.nNoise = c.nNoise;
    A.r = c.p.r;
    A.M = c.p.M;
    A.g = c.p.g;
    A.tol = c.p.cgTol;
    A.stopScale = c.eoStopScale;
    A.fac = -c.p.g * (c.p.driftMode == 1 ? c.p.cutFraction * c.p.cutFraction : 1.0);
    A.mode = c.p.cgTolMode;
    A.maxIter = c.p.cgMaxIter;
    A.maxRestarts = 4;
    // one entry per thread where the threads suffice (more waves for the same work), else two
    const int K = A.Vh <= kOnchipEoThreads ? 1 : 2;
    const int threads = (A.Vh / K + kWave - 1) / kWave * kWave;
    auto go = [&](auto kTag) {
        constexpr int KK = decltype(kTag)::value;
        auto *k = A.r == 1.0 ? &k_onchip_eo<KK, true, GEN, PROP> : &k_onchip_eo<KK, false, GEN, PROP>;
        hipLaunchKernelGGL(k, dim3(nsys), dim3(threads), 2 * EoLds<KK>::bytes, c.stream, A, phi,
                           (const uint64_t *)c.seed_d, streamBase, step, c.eta, bg, drift, out, c.cg_d, ratioIn, ratioOut,
                           nsys);
    };
    if (K == 1)
        go(std::integral_constant<int, 1>());
    else
        go(std::integral_constant<int, 2>());
    YCN_HIP(hipGetLastError());
    return YCN_OK;
}

int onchip_eo_force(Ctx &c, const double *phi, uint32_t streamBase, uint64_t step, bool chained) {
    const bool learn = c.p.cgTolMode == YCN_TOL_REL_TRUE && c.ratio;
    const size_t row = (size_t)c.nSys + 1;
    const double *in = learn && chained ? c.ratio + row * c.ratioTurn : nullptr;
    double *out = nullptr;
    if (learn) {
        c.ratioTurn ^= 1;
        out = c.ratio + row * c.ratioTurn;
    }
    const int rc = launch_eo<true, false>(c, phi, c.nSys, streamBase, step, c.t, onchip_share(c), nullptr, in, out);
    return rc ? rc : onchip_mean(c);
}

int onchip_eo_propagator(Ctx &c, const double *phi, double2 *out) {
    // (b_e in Ap: the measurement's out is t)
    return launch_eo<false, true>(c, phi, 1, 0, 0, c.Ap, nullptr, out, nullptr, nullptr);
}

}  // namespace ycn
