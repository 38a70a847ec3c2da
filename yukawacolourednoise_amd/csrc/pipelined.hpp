// pipelined.hpp -- the parts that the pipelined iterations share (plain.hip, eo_pipelined.hip,
// evenodd.hip): finalize kernels and stop decisions of both precisions, the FP32 ones' reliable
// update and host loop over chunks of launches, the FP64 ones' close.
#pragma once
#include <algorithm>
#include <type_traits>
#include <vector>

#include "cg_fused.hpp"
#include "cg_host.hpp"
#include "ycn_device.hpp"
#include "ycn_internal.hpp"

namespace ycn {

constexpr int kPfNT = 256;

// element idx of a buffer through a 32-bit byte offset (the buffers of one system are
// below 4 GiB), so that the load or store takes a scalar base and a vector offset
template <typename T>
__device__ __forceinline__ T &at(T *base, unsigned idx) {
    using C = typename std::conditional<std::is_const<T>::value, const char, char>::type;
    return *reinterpret_cast<T *>(reinterpret_cast<C *>(base) + (unsigned)(idx * (unsigned)sizeof(T)));
}

// a site's packed spinor: spins 0 and 1, each (flavour 0, flavour 1)
template <typename R>
struct Sp {
    typename Vec2<R>::T a, b;
};
// n of them in LDS, read and written without bank conflicts: whole 16-byte entries in FP32, a
// plane per spin in FP64
template <typename R, int N>
struct SpLds;
template <int N>
struct SpLds<float, N> {
    float4 e[N];
    __device__ __forceinline__ Sp<float> get(int i) const {
        const float4 v = e[i];
        return {make_float2(v.x, v.y), make_float2(v.z, v.w)};
    }
    __device__ __forceinline__ float2 s0(int i) const { return reinterpret_cast<const float2 *>(e)[2 * i]; }
    __device__ __forceinline__ float2 s1(int i) const { return reinterpret_cast<const float2 *>(e)[2 * i + 1]; }
    __device__ __forceinline__ void set(int i, Sp<float> v) { e[i] = make_float4(v.a.x, v.a.y, v.b.x, v.b.y); }
};
template <int N>
struct SpLds<double, N> {
    double2 e[2][N];
    __device__ __forceinline__ Sp<double> get(int i) const { return {e[0][i], e[1][i]}; }
    __device__ __forceinline__ double2 s0(int i) const { return e[0][i]; }
    __device__ __forceinline__ double2 s1(int i) const { return e[1][i]; }
    __device__ __forceinline__ void set(int i, Sp<double> v) {
        e[0][i] = v.a;
        e[1][i] = v.b;
    }
};

template <typename R>
__device__ __forceinline__ double sq(Sp<R> v) {
    return (double)((v.a.x * v.a.x + v.a.y * v.a.y) + (v.b.x * v.b.x + v.b.y * v.b.y));
}
template <typename R>
__device__ __forceinline__ Sp<R> axpy(Sp<R> u, R s, Sp<R> v) {
    return {mk2<R>(u.a.x + s * v.a.x, u.a.y + s * v.a.y), mk2<R>(u.b.x + s * v.b.x, u.b.y + s * v.b.y)};
}
// a spinor of two planes of V entries
template <typename R, typename P>
__device__ __forceinline__ Sp<R> load_sp(P *v, unsigned V, unsigned i) {
    return {at(v, i), at(v, V + i)};
}
template <typename R, typename P>
__device__ __forceinline__ void store_sp(P *v, unsigned V, unsigned i, Sp<R> s) {
    at(v, i) = s.a;
    at(v, V + i) = s.b;
}

// a mod n in [0, n) without an integer division (the 4-site halo of a tile spans several
// periods when an extent is smaller than 4, Nt = 2).  For |a| < 2^22 and inv = fl(1 / n),
// (a + 1/2) / n lies at least 1 / (2n) from an integer and the two single-precision
// roundings move it by less than |a + 1/2| / n * 2^-23, so the floor is exact.
__device__ __forceinline__ int wrapf(int a, int n, float inv) {
    return a - n * (int)floorf(((float)a + 0.5f) * inv);
}
__device__ __forceinline__ double2 pf_fin_sum(const double2 *part, int nb, double2 *lds) {
    double2 acc = make_double2(0.0, 0.0);
    int i = threadIdx.x;
    for (; i + 7 * kPfNT < nb; i += 8 * kPfNT) {
        double2 v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = part[i + u * kPfNT];
#pragma unroll
        for (int u = 0; u < 8; ++u) acc = cadd(acc, v[u]);
    }
    for (; i < nb; i += kPfNT) acc = cadd(acc, part[i]);
    return block_sum2<kPfNT>(acc, lds);
}

// ---------------------------------------------------------------------------
// finalize of the pipelined FP32 iteration
// ---------------------------------------------------------------------------
// the sums a launch leaves: mu = <p, Ap>, nu = |Ap|^2, rho = |r|^2
struct Pf3 {
    double mu, nu, rho;
};
// v of the lanes a permute swaps: lanes 32 .. 63 of a with lanes 0 .. 31 of b (HALF), or the odd
// rows of 16 of a with the even rows of b; the sum of the two afterwards
template <bool HALF>
__device__ __forceinline__ double swap_add(double a, double b) {
    const long long ia = __double_as_longlong(a), ib = __double_as_longlong(b);
    auto sw = [](unsigned u, unsigned v) {
        if constexpr (HALF)
            return __builtin_amdgcn_permlane32_swap(u, v, false, false);
        else
            return __builtin_amdgcn_permlane16_swap(u, v, false, false);
    };
    const auto lo = sw((unsigned)ia, (unsigned)ib), hi = sw((unsigned)(ia >> 32), (unsigned)(ib >> 32));
    return __longlong_as_double(((long long)hi[0] << 32) | lo[0]) +
           __longlong_as_double(((long long)hi[1] << 32) | lo[1]);
}
// Sums over the block by one barrier, valid in wave 0: mu, nu, rho in every lane of its rows of 16
// lanes 0, 1, 2.  The three sums share their steps: two swaps of lanes between registers leave each
// in rows of its own, four steps within rows finish them (7 additions and 14 moves against 18 and
// 52 for three separate sums).  red holds 3 NT / 64 numbers.
template <int NT>
__device__ __forceinline__ double block_sum3(double mu, double nu, double rho, double *red) {
    constexpr int NW = NT / kWave;
    static_assert(NW <= 16, "one row of lanes adds up the waves");
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave, row = lane >> 4, k = lane & 15;
    const double v = row_sum(swap_add<false>(swap_add<true>(mu, nu), swap_add<true>(rho, rho)));   // mu, rho, nu, rho
    if (k == 0 && row < 3) red[3 * wave + (row == 0 ? 0 : 3 - row)] = v;
    __syncthreads();
    return wave == 0 ? row_sum(row < 3 && k < NW ? red[3 * k + row] : 0.0) : 0.0;
}
// one system's nb block partials (pp[2 b] = (mu, nu), pp[2 b + 1].x = rho): the first loads, issued
// ahead of other work, and the sums by one block in a fixed order (thread t adds entries t, t + NT,
// ...; each round issues its U loads before adding); valid in wave 0
template <int NT>
struct PfParts {
    static constexpr int U = 4;
    double2 mn[U];
    double rh[U];
    __device__ __forceinline__ void load(const double2 *pp, int nb, int base) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = base + u * NT;
            mn[u] = make_double2(0.0, 0.0);
            rh[u] = 0.0;
            if (k < nb) {
                mn[u] = pp[2 * k];
                rh[u] = pp[2 * k + 1].x;
            }
        }
    }
    __device__ __forceinline__ void load(const double2 *pp, int nb) { load(pp, nb, threadIdx.x); }
    __device__ __forceinline__ Pf3 sum(const double2 *pp, int nb, double *red) {
        double mu = 0.0, nu = 0.0, rho = 0.0;
        for (int base = threadIdx.x;;) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                mu += mn[u].x;
                nu += mn[u].y;
                rho += rh[u];
            }
            base += U * NT;
            if (base - (int)threadIdx.x >= nb) break;
            load(pp, nb, base);
        }
        const double s = block_sum3<NT>(mu, nu, rho, red);
        return {lane_f64(s, 0), lane_f64(s, 16), lane_f64(s, 32)};
    }
};
template <int NT>
__device__ __forceinline__ Pf3 sum_pf_partials(const double2 *pp, int nb, double *red) {
    PfParts<NT> q;
    q.load(pp, nb);
    return q.sum(pp, nb, red);
}
// a block's own partials
template <int NT>
__device__ __forceinline__ void store_pf_partials(double2 *pp, double mu, double nu, double rho, double *red) {
    const double v = block_sum3<NT>(mu, nu, rho, red);
    if (threadIdx.x < 48 && (threadIdx.x & 15) == 0) reinterpret_cast<double *>(pp)[threadIdx.x >> 4] = v;
}

// what a launch reads of the state, none of it written while the launch runs except done
struct PfHead {
    double alpha, beta, stop, rrRel, rr;
    int iter0, maxIter, even, done;
};
__device__ __forceinline__ PfHead pf_head(const CgState &S) {
    return {S.alpha.x, S.beta, S.stop, S.rrRel, S.rr, S.iter0, S.maxIter, S.even, S.done};
}

// The decision after iteration number `iter` of the pipelined iteration, from (mu, nu)
// and the exact rho of that iteration: alpha = rho / mu and beta = (alpha^2 nu - rho) /
// rho for the next one (a negative prediction, from cancellation, restarts the
// direction).  Pause at the stop after an even number of iterations (the last direction
// applied is then in p[1]), at the cap, or on a non-positive <p, Ap>; a reliable update
// follows a pause.
struct PfStep {
    double alpha, beta;
    bool stop;
};
__device__ __forceinline__ PfStep pf_decide(const Pf3 &s, int iter, const PfHead &S) {
    const double mu = s.mu, nu = s.nu, rho = s.rho;
    PfStep d;
    d.stop = (iter >= S.maxIter) || (sqrt(rho) <= S.stop && !(iter & 1)) || (!(mu > 0.0) && !(iter & 1)) ||
             (rho < kReliableDrop * kReliableDrop * S.rrRel && !(iter & 1)) || !isfinite(mu) || !isfinite(rho);
    d.alpha = (mu > 0.0) ? rho / mu : 0.0;
    double rhoNext = d.alpha * d.alpha * nu - rho;
    if (!(rhoNext > 0.0)) rhoNext = 0.0;
    d.beta = (rho > 0.0) ? rhoNext / rho : 0.0;
    return d;
}

// the finalize of one iteration from its sums (thread 0): iteration count, rho, pause or
// the next alpha, beta; commit = false only keeps the sums (timing launches)
__device__ __forceinline__ void pf_commit(CgState &S, const Pf3 &s, int *active, int commit) {
    if (!commit) {
        S.rz = s.mu + s.nu + s.rho;   // a field these iterations never read
        return;
    }
    S.iter += 1;
    const PfStep d = pf_decide(s, S.iter, pf_head(S));
    S.rr_prev = S.rr;
    S.rr = s.rho;
    if (d.stop) {
        S.done = 1;
        atomicSub(active, 1);
        return;
    }
    S.alpha = make_double2(d.alpha, 0.0);
    S.beta = d.beta;
}

// The prologue of launch idx of a chunk (finMode 1; 2: timing, neither pausing nor writing the
// state): every block sums launch idx - 1's block partials (prevPart) in the same fixed order and
// derives the same alpha, beta and stop decision; a stopping launch's block 0 records the pause,
// with rho of the iteration before it from launch idx - 2's partials, still in this launch's own
// slot.  False: the system pauses here.  finMode 0 and launch 0 take alpha, beta from the state.
template <int NT>
__device__ __forceinline__ bool pf_prologue(CgState *st, const PfHead &hd, int sys, int idx, int finMode,
                                            PfParts<NT> &parts, const double2 *prevPart, const double2 *ownPart,
                                            int *active, double *red, double *bc, int *pause, double &alpha,
                                            double &beta) {
    alpha = hd.alpha;
    beta = hd.beta;
    if (finMode == 0 || idx == 0) return true;
    const int nb = (int)gridDim.x;
    const Pf3 s = parts.sum(prevPart + 2 * (size_t)sys * nb, nb, red);
    if (threadIdx.x == 0) {
        const PfStep d = pf_decide(s, hd.iter0 + idx, hd);
        bc[0] = d.alpha;
        bc[1] = d.beta;
        *pause = finMode == 1 && d.stop;
    }
    __syncthreads();
    if (!*pause) {
        alpha = bc[0];
        beta = bc[1];
        return true;
    }
    if (blockIdx.x == 0) {
        double rprev = hd.rr;   // iteration iter0 (chunk start) when idx == 1
        if (idx >= 2) {
            __syncthreads();
            rprev = sum_pf_partials<NT>(ownPart + 2 * (size_t)sys * nb, nb, red).rho;
        }
        if (threadIdx.x == 0) {
            CgState &S = st[sys];
            S.iter = S.iter0 + idx;
            S.rr_prev = rprev;
            S.rr = s.rho;
            S.done = 1;
            atomicSub(active, 1);
        }
    }
    return false;
}

// ---------------------------------------------------------------------------
// finalize of the pipelined FP64 iterations
// ---------------------------------------------------------------------------
// The decision after a launch that would complete iteration number `iter` of the textbook
// recurrence (its r update included): alpha, and |r|^2 after it from the recurrence.  That
// prediction is off by a few eps rho, so it is not taken below 1e-13 rho; and where rho itself,
// summed exactly, has reached the stop, the step is not taken.  Stop as the unpipelined
// iteration does (k_fin_beta): at the stop (after an even number of iterations where S.even), at
// the cap, or on a NaN.
struct P64Step {
    double alpha, beta, rr;
    int iter;
    bool stop, conv;
};
__device__ __forceinline__ P64Step p64_decide(const Pf3 &s, int iter, const PfHead &S) {
    const double mu = s.mu, nu = s.nu, rho = s.rho;
    P64Step d;
    if (sqrt(rho) <= S.stop && !(S.even && !(iter & 1) && rho > 0.0)) return {0.0, 0.0, rho, iter - 1, true, true};
    d.iter = iter;
    d.alpha = rho / mu;
    d.rr = d.alpha * d.alpha * nu - rho;
    if (d.rr <= 1e-13 * rho) d.rr = 1e-13 * rho;
    d.beta = d.rr / rho;
    d.conv = sqrt(d.rr) <= S.stop;
    d.stop = (!(sqrt(d.rr) > S.stop) && !(S.even && (iter & 1))) || iter >= S.maxIter;
    return d;
}
// a system stops after the launch that iteration `it` names, its last x updates left to the close
__device__ __forceinline__ void p64_stop(CgState &S, int it, const P64Step &d, int *active) {
    S.done = 1;
    S.converged = d.conv ? 1 : 0;
    S.pfLaunch = it - S.pfBase;
    atomicSub(active, 1);
}

// pf_prologue for FP64
template <int NT>
__device__ __forceinline__ bool p64_prologue(CgState *st, const PfHead &hd, int sys, int idx, int finMode,
                                             PfParts<NT> &parts, const double2 *prevPart, int *active, double *red,
                                             double *bc, int *pause, double &alpha, double &beta) {
    alpha = hd.alpha;
    beta = hd.beta;
    if (finMode == 0 || idx == 0) return true;
    const int nb = (int)gridDim.x;
    const Pf3 s = parts.sum(prevPart + 2 * (size_t)sys * nb, nb, red);
    if (threadIdx.x == 0) {
        const int it = hd.iter0 + idx;
        const P64Step d = p64_decide(s, it, hd);
        bc[0] = d.alpha;
        bc[1] = d.beta;
        *pause = finMode == 1 && d.stop;
        if (finMode == 1 && d.stop && blockIdx.x == 0) {
            CgState &S = st[sys];
            S.alpha = make_double2(d.alpha, 0.0);
            S.beta = d.beta;
            S.iter = d.iter;
            S.rr_prev = s.rho;
            S.rr = d.rr;
            p64_stop(S, it, d, active);
        }
    }
    __syncthreads();
    alpha = bc[0];
    beta = bc[1];
    return !*pause;
}

// Finalize after the launches of a chunk that finalized each other (n of them), or after one
// launch (n = 1); commit = 0 only reduces (timing).
template <int NT>
__global__ void __launch_bounds__(NT)
k_fin_p64(const double2 *__restrict__ part, int nb, int n, CgState *__restrict__ st, int *__restrict__ active,
          int commit) {
    __shared__ double red[3 * NT / kWave];
    CgState &S = st[blockIdx.x];
    const PfHead hd = pf_head(S);
    const Pf3 s = sum_pf_partials<NT>(part + 2 * (size_t)blockIdx.x * nb, nb, red);
    if (hd.done || threadIdx.x) return;
    if (!commit) {
        S.rz = s.mu + s.nu + s.rho;   // a field these iterations never read
        return;
    }
    const P64Step d = p64_decide(s, hd.iter0 + n, hd);
    S.alpha = make_double2(d.alpha, 0.0);
    S.beta = d.beta;
    S.iter = d.iter;
    S.rr_prev = s.rho;
    S.rr = d.rr;
    S.iter0 += n;
    if (d.stop) p64_stop(S, S.iter0, d, active);
}

inline void launch_fin_p64(Ctx &c, int nsys, int nb, int n, const double2 *part, int commit) {
    if (nb > 4 * kPfNT)
        hipLaunchKernelGGL(k_fin_p64<1024>, dim3(nsys), dim3(1024), 0, c.stream, part, nb, n, c.cg_d, c.active, commit);
    else
        hipLaunchKernelGGL(k_fin_p64<kPfNT>, dim3(nsys), dim3(kPfNT), 0, c.stream, part, nb, n, c.cg_d, c.active,
                           commit);
}

// the separate finalize of one iteration (one block per system, after a finMode 0
// launch); commit = false only reduces (timing)
template <int NT>
__global__ void __launch_bounds__(NT)
k_fin_pf(const double2 *__restrict__ part, int nb, CgState *__restrict__ st, int *__restrict__ active, int commit) {
    __shared__ double red[3 * NT / kWave];
    CgState &S = st[blockIdx.x];
    const int skip = S.done;
    const Pf3 s = sum_pf_partials<NT>(part + 2 * (size_t)blockIdx.x * nb, nb, red);
    if (skip || threadIdx.x) return;
    pf_commit(S, s, active, commit);
}

// the same with one wave per system (systems with at most kPfNT block partials: one or a
// few loads per lane and a shuffle reduction, no LDS or barriers)
static __global__ void __launch_bounds__(kPfNT)
k_fin_pf_wave(const double2 *__restrict__ part, int nb, int nsys, CgState *__restrict__ st, int *__restrict__ active,
              int commit) {
    const int sys = blockIdx.x * (kPfNT / kWave) + (int)threadIdx.x / kWave;
    const int lane = threadIdx.x & (kWave - 1);
    if (sys >= nsys) return;
    CgState &S = st[sys];
    const int skip = S.done;
    const double2 *pp = part + 2 * (size_t)sys * nb;
    double mu = 0.0, nu = 0.0, rho = 0.0;
    for (int k = lane; k < nb; k += kWave) {
        const double2 mn = pp[2 * k];
        mu += mn.x;
        nu += mn.y;
        rho += pp[2 * k + 1].x;
    }
    const Pf3 s = {wave_sum(mu), wave_sum(nu), wave_sum(rho)};
    if (skip || lane) return;
    pf_commit(S, s, active, commit);
}

// one wave per system for few partials, 1024 threads once a system has more partials
// than four rounds of 256 threads cover
inline void launch_fin_pf(Ctx &c, int nsys, int nb, int commit, const double2 *part) {
    if (nb <= kPfNT)
        hipLaunchKernelGGL(k_fin_pf_wave, dim3((nsys + kPfNT / kWave - 1) / (kPfNT / kWave)), dim3(kPfNT), 0, c.stream,
                           part, nb, nsys, c.cg_d, c.active, commit);
    else if (nb > 4 * kPfNT)
        hipLaunchKernelGGL(k_fin_pf<1024>, dim3(nsys), dim3(1024), 0, c.stream, part, nb,
                           c.cg_d, c.active, commit);
    else
        hipLaunchKernelGGL(k_fin_pf<kPfNT>, dim3(nsys), dim3(kPfNT), 0, c.stream, part, nb,
                           c.cg_d, c.active, commit);
}

// reliable update of the pipelined iteration: x += x_s (FP64), x_s = 0, and the last
// direction applied copied to p[0], where the next chunk's launch 0 reads it.  After m
// launches (m counted from the state per system) that is p_{m-2}, in rotation slot
// (m - 1) mod 3 of p[0], p[1], p2.  For odd m (a stop at the iteration cap after an even
// launch) the even launch's deferred term alpha_{m-1} p_{m-2} is added too, with the alpha
// it recorded in ab.
[[maybe_unused]] static __global__ void __launch_bounds__(kPfNT)
k_pf_reliable(int n, int chunk, const CgState *__restrict__ st, double2 *__restrict__ x, float2 *__restrict__ xs,
              const float2 *__restrict__ p1, const float2 *__restrict__ p2, float2 *__restrict__ p0) {
    const int sys = blockIdx.y;
    if (st[sys].final_) return;
    const int s = blockIdx.x * kPfNT + threadIdx.x;
    if (s >= n) return;
    // (a chunk of prologue-finalized launches that no stop has ended is still to be recorded)
    const int m = chunk && !st[sys].done ? chunk : st[sys].iter - st[sys].iter0, slot = m >= 1 ? (m - 1) % 3 : 0;
    const float2 *src = slot == 1 ? p1 : slot == 2 ? p2 : p0;
    const double a = (m & 1) ? st[sys].ab[(m - 1) & 1].x : 0.0;
    const size_t off = (size_t)sys * 2 * n;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
        const size_t i = off + (size_t)c * n + s;
        const float2 d = xs[i];
        const double2 xv = x[i];
        double2 xn = make_double2(xv.x + (double)d.x, xv.y + (double)d.y);
        const float2 pk = (slot != 0 || (m & 1)) ? src[i] : make_float2(0.f, 0.f);
        if (m & 1) xn = make_double2(xn.x + a * (double)pk.x, xn.y + a * (double)pk.y);
        x[i] = xn;
        xs[i] = make_float2(0.f, 0.f);
        if (slot != 0) p0[i] = pk;
    }
}

// What ends a chunk of n launches that finalized each other in their prologues: launch n - 1's
// partials in slot 1, launch n - 2's in slot 0 (n is even), nb per system.  n = 0: a finalize launch
// followed each.
struct PfChunkEnd {
    int n, nb;
    const double2 *last, *before;
};
inline PfChunkEnd pf_chunk_end(const Ctx &c, int n) {
    if (!c.eoFinFused) return {0, 0, nullptr, nullptr};
    return {n, c.eoPfBlocks, c.pfSlot[1], c.pfSlot[0]};
}

// The decision that ends a chunk, and the one after its reliable update, one block per system.  The
// first takes the place of a prologue after launch n - 1 (end.n > 0; systems that paused inside the
// chunk already hold their state).  Reliable update: partRes = |b_e - S x_e|^2 and
// partN = |S^T (b_e - S x_e)|^2 (the new normal residual).  Converged on the system residual, or resume with alpha = 0 (r already is the true
// residual) and beta = |r_true|^2 / |r_prev|^2 (the direction is kept)
[[maybe_unused]] static __global__ void __launch_bounds__(kPfNT)
k_fin_pf_true(const double2 *__restrict__ partRes, const double2 *__restrict__ partN, int nb,
                 CgState *__restrict__ st, int *__restrict__ active, PfChunkEnd end) {
    __shared__ double2 lds0[kPfNT / kWave], lds1[kPfNT / kWave];
    __shared__ double red[2][3 * kPfNT / kWave];
    const int sys = blockIdx.x;
    const int skip = st[sys].final_, paused = st[sys].done;
    if (skip) return;
    Pf3 s{}, before{};
    if (end.n && !paused) {
        s = sum_pf_partials<kPfNT>(end.last + 2 * (size_t)sys * end.nb, end.nb, red[0]);
        before = sum_pf_partials<kPfNT>(end.before + 2 * (size_t)sys * end.nb, end.nb, red[1]);
    }
    const double2 res = pf_fin_sum(partRes + (size_t)sys * nb, nb, lds0);
    const double2 rn = pf_fin_sum(partN + (size_t)sys * nb, nb, lds1);
    if (threadIdx.x) return;
    CgState &S = st[sys];
    if (end.n && !paused) {
        S.iter = S.iter0 + end.n;
        S.rr_prev = before.rho;
        S.rr = s.rho;
        if (pf_decide(s, S.iter, pf_head(S)).stop) {
            S.done = 1;
            atomicSub(active, 1);
        }
    }
    S.true_rel = S.enorm2 > 0.0 ? sqrt(res.x / S.enorm2) : sqrt(res.x);
    S.restarts += 1;
    if (S.nRu < kMaxRounds) S.ruIter[S.nRu] = S.iter;
    S.nRu += 1;
    // paused at the stop (not for the drop since the last anchor): the normal-equation
    // threshold the true residual asks for
    if (S.done && sqrt(S.rr) <= S.stop && S.true_rel > 0.0) S.need = sqrt(rn.x) * S.tol / S.true_rel;
    const bool conv = (S.mode == YCN_TOL_REL_TRUE) ? (S.true_rel <= S.tol) : (sqrt(rn.x) <= S.stop);
    if (conv || S.iter >= S.maxIter) {
        S.converged = conv ? 1 : 0;
        S.final_ = 1;
        if (!S.done) {
            S.done = 1;
            atomicSub(active, 1);
        }
        return;
    }
    S.alpha = make_double2(0.0, 0.0);
    S.beta = (S.rr_prev > 0.0) ? rn.x / S.rr_prev : 0.0;
    S.rr = rn.x;
    S.rrRel = rn.x;
    S.iter0 = S.iter;   // the next chunk's launches count from here
    if (S.mode == YCN_TOL_REL_TRUE && sqrt(rn.x) <= S.stop) S.stop = sqrt(rn.x) * 0.5 * S.tol / S.true_rel;
    if (S.done) {
        S.done = 0;
        atomicAdd(active, 1);
    }
}

constexpr int kP64Launches = 12;   // per captured FP64 chunk: keeps the rotations of both buffer sets

// The x updates that the launches of an FP64 phase have left to later ones, added to x of the
// systems that stopped after m = pfLaunch launches: alpha_{m-1} p_{m-1}, and after an odd number
// of launches alpha_{m-2} p_{m-2} before it.  d0, d1, d2: the directions' rotation, p_{-1} in d0
// and the phase's first r in d2.  KEEP: the next phase goes on from here, so r (into d2) and the
// direction (into d0) are brought up too, from the A p of even (a0) and odd (a1) launches.
template <bool KEEP>
__global__ void __launch_bounds__(kPfNT)
k_p64_close(int n, const CgState *__restrict__ st, double2 *__restrict__ x, double2 *__restrict__ d0,
            const double2 *__restrict__ d1, double2 *__restrict__ d2, const double2 *__restrict__ a0,
            const double2 *__restrict__ a1) {
    const int sys = blockIdx.y, m = st[sys].pfLaunch, i = blockIdx.x * kPfNT + threadIdx.x;
    if (m == 0 || i >= n) return;
    const double al = st[sys].alpha.x;
    const double2 ab = st[sys].ab[(m - 1) & 1];   // of launch m - 1: alpha_{m-2}, beta_{m-1}
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const size_t k = ((size_t)sys * 2 + s) * n + i;
        const double2 v0 = d0[k], v1 = d1[k], v2 = d2[k];
        const double2 p = m % 3 == 0 ? v0 : m % 3 == 1 ? v1 : v2, pp = m % 3 == 0 ? v2 : m % 3 == 1 ? v0 : v1;
        double2 v = x[k];
        if ((m & 1) && m > 1) v = make_double2(v.x + ab.x * pp.x, v.y + ab.x * pp.y);
        x[k] = make_double2(v.x + al * p.x, v.y + al * p.y);
        if (KEEP) {
            const double2 q = (m & 1) ? a0[k] : a1[k];
            const double2 rk = m == 1 ? v2 : make_double2(p.x - ab.y * pp.x, p.y - ab.y * pp.y);
            d2[k] = make_double2(rk.x - al * q.x, rk.y - al * q.y);
            d0[k] = p;
        }
    }
}

// a launch of the even-odd pipelined iteration (k_eo_pf)
template <typename R>
struct EoPfLaunch {
    using V2 = typename Vec2<R>::T;
    const R *phi;
    const V2 *r, *Ap_in, *pold;
    V2 *pnew, *Ap, *x;
    double2 *part;
    const double2 *prevPart;
    int idx, form, finMode;
    bool persist;
};
int launch_eo_pf32(const Ctx &c, int TT, int TX, int nsys, const EoPfLaunch<float> &b);
int launch_eo_pf64(const Ctx &c, int TT, int TX, int nsys, const EoPfLaunch<double> &b);

// blocks that the device holds of the kernel with the fewest of ks (persistent launches:
// consecutive ones then leave the same number of partials)
template <typename K>
inline int resident_blocks(const K (&ks)[3], int threads) {
    int dev = 0, cus = 0, m = 1 << 30;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return 8;
    for (const K &k : ks) {
        int per = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, reinterpret_cast<const void *>(k), threads, 0) !=
            hipSuccess)
            return 8;
        m = std::min(m, per * cus);
    }
    return std::max(m, 8);
}
// the grid: as many blocks as are resident, or fewer where that evens out the tiles per block; a
// multiple of 8, so that a block's tiles lie in one XCD's band of tiles
inline int persistent_grid(int resident, int tiles) {
    const int rounds = (tiles + resident - 1) / resident, g = (tiles + rounds - 1) / rounds;
    return std::min(tiles, (g + 7) / 8 * 8);
}

// direction p_k (k >= -1) of a chunk of pipelined launches: the three buffers in rotation,
// p_{-1} (the direction kept across the reliable update) in ps[0]
inline float2 *pf_dir(const Ctx &c, int k) {
    float2 *const rot[3] = {c.ps[0], c.ps[1], c.pfP2};
    return rot[(k + 1) % 3];
}

// Length of the next chunk: the reliable-update interval until the predicted iteration
// count is near, then just past it (a multiple of 8), so that few launches run after the
// systems have paused.
inline int pf_chunk_len(const Ctx &c, int pred, int itDone) {
    const int every = std::max(1, c.p.reliableEvery);
    const int nIt = every + (every & 1);
    const int rem = pred - itDone + 4;
    if (pred > 0 && rem < nIt) return std::max(8, (rem + 7) / 8 * 8);
    return nIt;
}

// the eager loop polls once it is within this many iterations of the prediction
inline int pf_poll_margin(int pred) { return std::max(8, pred / 8); }

// The pipelined FP32 solve from the state the setup (or an unfinished enqueued solve)
// left, until every system is final, polling the systems only where they may have
// converged; itDone: iterations already done (the chunk lengths count from there).
// The summary goes to *st, the iteration count and the starting threshold of the next
// solve are learned from it.
// chunk(n): n launches of the iteration and the reliable update that closes them.
template <typename Chunk>
inline int pf_loop(Ctx &c, int nsys, int itDone, SolveStats *st, Chunk chunk) {
    const int every = std::max(1, c.p.reliableEvery);
    const int nIt = every + (every & 1);
    const int hardCap = c.p.cgMaxIter + nIt + 8;
    int launched = 0, active = nsys, rc;
    // profiling the iteration with the prologue finalize: a chunk is nothing but
    // back-to-back iteration launches, so one event pair brackets it and its working
    // launches are the iterations the systems did in it (the most of any system)
    const bool chunkProf = c.profTarget == PK_NORMAL_OP && c.eoFinFused;
    std::vector<int> itPrev(chunkProf ? nsys : 0, 0);
    bool polled = true;
    while (active > 0 && launched < hardCap) {
        const int n = pf_chunk_len(c, c.eoPredIters, itDone);
        const int slot = chunkProf ? prof_chunk_begin(c, PK_NORMAL_OP) : -1;
        rc = chunk(n);
        prof_chunk_end(c, slot);
        if (rc) return rc;
        launched += n;
        // poll only where the systems may have converged: well short of the previous
        // solve's iteration count they cannot have, so the next chunk is enqueued at
        // once (its kernels exit at once for systems that are final after all)
        if (c.eoPredIters > 0 && itDone + n + pf_poll_margin(c.eoPredIters) < c.eoPredIters && !chunkProf) {
            itDone += n;
            polled = false;
            continue;
        }
        rc = poll_iters(c, nsys, active, itDone);
        if (rc) return rc;
        polled = true;
        if (chunkProf) {
            int work = 0;
            for (int k = 0; k < nsys; ++k) {
                work = std::max(work, c.cg_h[k].iter - itPrev[k]);
                itPrev[k] = c.cg_h[k].iter;
            }
            if (slot >= 0) c.evWork[slot] = work;
        }
    }
    if (!polled) {   // the launch cap ended the loop after a skipped poll
        rc = poll_iters(c, nsys, active, itDone);
        if (rc) return rc;
    }
    SolveStats out;   // the last poll left the final states in the mirror
    rc = stats_from_mirror(c, nsys, &out);
    if (rc) return rc;
    c.eoPredIters = out.iters_max;
    int kMax = 0;
    for (int k = 1; k < nsys; ++k)
        if (c.cg_h[k].iter > c.cg_h[kMax].iter) kMax = k;
    c.eoRounds.assign(c.cg_h[kMax].ruIter, c.cg_h[kMax].ruIter + std::min(c.cg_h[kMax].nRu, kMaxRounds));
    if (st) *st = out;
    return YCN_OK;
}

}  // namespace ycn
