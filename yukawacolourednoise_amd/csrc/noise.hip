// noise.hip -- coloured noise on gfx950 (replaces ColouredNoise,
// code/src/colouredNoise.cpp:16-29,40-67,138-178, and its cuFFT D2Z/Z2D calls).
//
// Mixed-radix Stockham FFTs in LDS (radix 8, 4, 2, 3, 5 and 7 butterflies in registers,
// any other prime by a direct DFT), in three passes:
//   rows_fwd : Philox N(0,1) field generated in registers, rows t and t+1 packed as
//              z = xi_t + i xi_{t+1}, forward FFT along x, untangled into the two
//              half spectra -> spec[rep][t][kx]
//   cols     : each kx column: forward FFT along t, mask (kx <= kmax[kt] ? 1/V : 0),
//              inverse FFT along t, in place
//   rows_inv : rows t, t+1 re-packed with the Hermitian extension (C2R convention:
//              imaginary parts of the kx = 0 and kx = Nx/2 bins are ignored), inverse
//              FFT along x, real/imag parts -> noise rows t, t+1
// Columns beyond the cutoff, kx > kmaxAll, are neither written, transformed nor read: with
// cutoff s about a share s sqrt(2) of them is kept.  A lattice whose half spectrum fits LDS
// takes one block per replica and one launch for everything.
// Algorithmic HBM traffic ~ 8 (rows_fwd write) + 16 (cols r/w) + 8 + 8 (rows_inv)
// = 40 bytes per site.
//
// What bounds it is latency: at 1024 x 1024 a pass holds 512 lines of 1024 points, four to eight
// waves per CU, and each FFT pass is a chain of an LDS read, a twiddle load, a butterfly, an LDS
// write and a barrier.  So butterflies are of radix 8 and 4, whose instructions spread over the
// block's lanes (a radix-16 one is 660 instructions of one lane, and 64 of them hold a line of
// 1024), a thread requests all it needs from memory before it waits, blocks have a thread per two
// points, index divisions are multiplications and LDS rows are padded against power-of-two strides.
// A field into a device buffer, before these choices (radix 16, eight points per thread, a load at a
// time) and with them: 1024 x 1024 50.0 -> 43.6 us (columns 18, rows forward 13, rows inverse 9),
// 512 x 512 36.9 -> 27.8, 256 x 256 42.3 -> 24.8, four of 256 x 480 45.9 -> 30.7.
#include <math.h>

#include <algorithm>
#include <mutex>
#include <vector>

#include "ycn_device.hpp"
#include "ycn_internal.hpp"

namespace ycn {

constexpr int kFftThreads = 256;
constexpr int kLineThreads = 512;   // most threads of a block of the line passes
// The launches never fill a SIMD with more than four waves: registers for loads in flight instead
// (left to itself the compiler keeps to 62 of 128 and waits for each load: 512 x 512 34.9 us a
// field against 27.8)
#define YCN_FOUR_WAVES __attribute__((amdgpu_waves_per_eu(4, 4)))
constexpr int kFftLdsBytes = 73760;  // two padded ping-pong buffers per block (one line of 2048)

// ---------------------------------------------------------------------------
// DFTs of one butterfly in registers, natural order in and out
// ---------------------------------------------------------------------------
// v times -i (forward) or +i (inverse)
template <bool INV>
__device__ __forceinline__ double2 rot(double2 v) {
    return INV ? make_double2(-v.y, v.x) : make_double2(v.y, -v.x);
}
// v times exp(-+ i phi), given (cos phi, sin phi)
template <bool INV>
__device__ __forceinline__ double2 twid(double2 v, double2 w) {   // w = exp(-i phi) from the table
    return INV ? make_double2(v.x * w.x + v.y * w.y, v.y * w.x - v.x * w.y) : cmul(v, w);
}
template <bool INV>
__device__ __forceinline__ void dft4(double2 &a, double2 &b, double2 &c, double2 &d) {
    const double2 t0 = cadd(a, c), t1 = csub(a, c), t2 = cadd(b, d), t3 = rot<INV>(csub(b, d));
    a = cadd(t0, t2);
    b = cadd(t1, t3);
    c = csub(t0, t2);
    d = csub(t1, t3);
}
// cos(2 pi k / R), sin(2 pi k / R) of the odd radices
template <int R> struct OddRoots;
template <> struct OddRoots<3> {
    static constexpr double c[3] = {1.0, -0.5, -0.5};
    static constexpr double s[3] = {0.0, 0.86602540378443864676, -0.86602540378443864676};
};
template <> struct OddRoots<5> {
    static constexpr double c[5] = {1.0, 0.30901699437494742410, -0.80901699437494742410, -0.80901699437494742410,
                                    0.30901699437494742410};
    static constexpr double s[5] = {0.0, 0.95105651629515357212, 0.58778525229247312917, -0.58778525229247312917,
                                    -0.95105651629515357212};
};
template <> struct OddRoots<7> {
    static constexpr double c[7] = {1.0, 0.62348980185873353053, -0.22252093395631440429, -0.90096886790241912624,
                                    -0.90096886790241912624, -0.22252093395631440429, 0.62348980185873353053};
    static constexpr double s[7] = {0.0, 0.78183148246802980871, 0.97492791218182360702, 0.43388373911755812048,
                                    -0.43388373911755812048, -0.97492791218182360702, -0.78183148246802980871};
};
template <int R, bool INV>
__device__ __forceinline__ void dft(double2 (&v)[R]) {
    if constexpr (R == 2) {
        const double2 a = v[0];
        v[0] = cadd(a, v[1]);
        v[1] = csub(a, v[1]);
    } else if constexpr (R == 4) {
        dft4<INV>(v[0], v[1], v[2], v[3]);
    } else if constexpr (R == 8) {
        constexpr double h = 0.70710678118654752440;
        dft4<INV>(v[0], v[2], v[4], v[6]);
        dft4<INV>(v[1], v[3], v[5], v[7]);
        v[3] = twid<INV>(v[3], make_double2(h, -h));
        v[5] = rot<INV>(v[5]);
        v[7] = twid<INV>(v[7], make_double2(-h, -h));
        double2 o[8];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            o[k] = cadd(v[2 * k], v[2 * k + 1]);
            o[k + 4] = csub(v[2 * k], v[2 * k + 1]);
        }
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] = o[k];
    } else {
        // odd prime: pairs q, R - q
        constexpr int M = (R - 1) / 2;
        double2 sm[M], df[M], o[R];
        o[0] = v[0];
#pragma unroll
        for (int q = 0; q < M; ++q) {
            sm[q] = cadd(v[q + 1], v[R - 1 - q]);
            df[q] = csub(v[q + 1], v[R - 1 - q]);
            o[0] = cadd(o[0], sm[q]);
        }
#pragma unroll
        for (int k = 1; k <= M; ++k) {
            double2 e = v[0], f = make_double2(0.0, 0.0);
#pragma unroll
            for (int q = 0; q < M; ++q) {
                e = cadd(e, cscl(OddRoots<R>::c[((q + 1) * k) % R], sm[q]));
                f = cadd(f, cscl(OddRoots<R>::s[((q + 1) * k) % R], df[q]));
            }
            f = rot<INV>(f);
            o[k] = cadd(e, f);
            o[R - k] = csub(e, f);
        }
#pragma unroll
        for (int k = 0; k < R; ++k) v[k] = o[k];
    }
}

// ---------------------------------------------------------------------------
// LDS Stockham FFT over `lines` lines of length n, element e of a line at fft_at(e) of its
// row of fft_row(n) entries: one entry of padding in eight, so that the first pass's stores
// at strides of the radix spread over the banks.
// ---------------------------------------------------------------------------
__host__ __device__ __forceinline__ int fft_at(int e) { return e + (e >> 3); }
__host__ __device__ __forceinline__ int fft_row(int n) { return n + (n >> 3) + 1; }
// a / n for 0 <= a < 2^22 with inv = 1 / n in single precision: (a + 1/2) / n lies at least
// 1 / (2n) from an integer and the roundings move it by less
__device__ __forceinline__ int fast_div(int a, float inv) { return (int)(((float)a + 0.5f) * inv); }

template <int R, bool INV>
__device__ __forceinline__ void fft_pass(const double2 *a, double2 *b, int lines, int row, const FftPass &F,
                                         const double2 *__restrict__ tw) {
    const int nb = F.nb, Ns = F.Ns, tstride = F.tstride;
    const float invNb = F.invNb, invNs = F.invNs;
    for (int w = threadIdx.x; w < nb * lines; w += blockDim.x) {
        const int line = fast_div(w, invNb), j = w - line * nb;
        const int jd = fast_div(j, invNs), jm = j - jd * Ns;
        const double2 *in = a + line * row;
        double2 *out = b + line * row;
        double2 v[R];
#pragma unroll
        for (int q = 0; q < R; ++q) v[q] = in[fft_at(j + q * nb)];
        if (jm) {
            const int ts = jm * tstride;
#pragma unroll
            for (int q = 1; q < R; ++q) v[q] = twid<INV>(v[q], tw[q * ts]);
        }
        dft<R, INV>(v);
        const int o = jd * Ns * R + jm;
#pragma unroll
        for (int k = 0; k < R; ++k) out[fft_at(o + k * Ns)] = v[k];
    }
}

// any other prime factor: one thread per output, a direct sum of R terms
template <bool INV>
__device__ void fft_pass_prime(const double2 *a, double2 *b, int lines, const FftPlan &P, const FftPass &F,
                               const double2 *__restrict__ tw) {
    const int n = P.n, R = F.R, Ns = F.Ns, nb = F.nb, tstride = F.tstride, row = fft_row(n);
    for (int w = threadIdx.x; w < n * lines; w += blockDim.x) {
        const int line = w / n, o = w - line * n;
        const int jd = o / (Ns * R), rem = o - jd * Ns * R, k = rem / Ns, jm = rem - k * Ns;
        const int j = jd * Ns + jm;
        const double2 *in = a + line * row;
        // exponent per input: the Stockham twiddle and the DFT kernel w_R^{qk}, modulo n
        const int step = (jm * tstride + k * nb) % n;
        double2 acc = in[fft_at(j)];
        int e = 0;
        for (int q = 1; q < R; ++q) {
            e += step;
            if (e >= n) e -= n;
            acc = cadd(acc, twid<INV>(in[fft_at(j + q * nb)], tw[e]));
        }
        b[line * row + fft_at(o)] = acc;
    }
}

// transforms a (barrier before and after); returns the buffer holding the result (a or b)
template <bool INV>
__device__ __forceinline__ double2 *lds_fft(double2 *a, double2 *b, int lines, const FftPlan &P, const double2 *tw) {
    const int row = fft_row(P.n);
    for (int f = 0; f < P.nf; ++f) {
        const FftPass &F = P.pass[f];
        switch (F.R) {
        case 8: fft_pass<8, INV>(a, b, lines, row, F, tw); break;
        case 4: fft_pass<4, INV>(a, b, lines, row, F, tw); break;
        case 2: fft_pass<2, INV>(a, b, lines, row, F, tw); break;
        case 3: fft_pass<3, INV>(a, b, lines, row, F, tw); break;
        case 5: fft_pass<5, INV>(a, b, lines, row, F, tw); break;
        case 7: fft_pass<7, INV>(a, b, lines, row, F, tw); break;
        default: fft_pass_prime<INV>(a, b, lines, P, F, tw); break;
        }
        __syncthreads();
        double2 *tmp = a;
        a = b;
        b = tmp;
    }
    return a;
}
template <bool INV>
__device__ __forceinline__ double2 *lds_fft(double2 *a, double2 *b, int lines, const FftPlan &P) {
    return lds_fft<INV>(a, b, lines, P, P.tw);
}

// Row pairs pair0 .. pair0 + np - 1 of the white field into the LDS lines a: from xi, or
// generated.  A Philox call gives the normals of two sites, which lie in one row when Nx is
// even: a thread then takes both.
__device__ __forceinline__ void load_rows(double2 *a, const double *__restrict__ xi, uint64_t seed, uint64_t step,
                                          int pair0, int np, int Nt, int Nx) {
    const int row = fft_row(Nx);
    if (!xi && Nx % 2 == 0) {
        const int Nh = Nx / 2;
        const float inv = 1.0f / (float)Nh;
        for (int w = threadIdx.x; w < np * Nh; w += blockDim.x) {
            const int l = fast_div(w, inv), x = 2 * (w - l * Nh);
            const int t0 = 2 * (pair0 + l);
            double2 g0 = make_double2(0.0, 0.0), g1 = g0;
            if (t0 < Nt) g0 = normal_pair(seed, 0u, step, ((uint64_t)t0 * Nx + x) >> 1);
            if (t0 + 1 < Nt) g1 = normal_pair(seed, 0u, step, ((uint64_t)(t0 + 1) * Nx + x) >> 1);
            a[l * row + fft_at(x)] = make_double2(g0.x, g1.x);
            a[l * row + fft_at(x + 1)] = make_double2(g0.y, g1.y);
        }
        return;
    }
    for (int w = threadIdx.x; w < np * Nx; w += blockDim.x) {
        const int l = w / Nx, x = w - l * Nx;
        double v[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int t = 2 * (pair0 + l) + u;
            const int64_t i = (int64_t)t * Nx + x;
            v[u] = 0.0;
            if (t < Nt) {
                if (xi) {
                    v[u] = xi[i];
                } else {
                    const double2 g = normal_pair(seed, 0u, step, (uint64_t)(i >> 1));
                    v[u] = (i & 1) ? g.y : g.x;
                }
            }
        }
        a[l * row + fft_at(x)] = make_double2(v[0], v[1]);
    }
}

// use(w, get(w)) for every w < n that is this thread's; U values are requested before any is used,
// so that a thread waits for memory once per U
template <int U, typename T, typename Get, typename Use>
__device__ __forceinline__ void batched(int n, Get get, Use use) {
    for (int base = threadIdx.x; base < n; base += U * blockDim.x) {
        T v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int w = base + u * blockDim.x;
            if (w < n) v[u] = get(w);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int w = base + u * blockDim.x;
            if (w < n) use(w, v[u]);
        }
    }
}

struct RowPair {
    double2 A, B;
};

// the half spectra of rows t0, t0 + 1 at column k from their packed transform (a line)
__device__ __forceinline__ void untangle(const double2 *line, int k, int Nx, double2 &A, double2 &B) {
    // A = (Z_k + conj Z_-k)/2 ; B = (Z_k - conj Z_-k)/(2i)
    const double2 zk = line[fft_at(k)], zm = line[fft_at(k == 0 ? 0 : Nx - k)];
    A = make_double2(0.5 * (zk.x + zm.x), 0.5 * (zk.y - zm.y));
    B = make_double2(0.5 * (zk.y + zm.y), -0.5 * (zk.x - zm.x));
}

// the packed line's entries k and Nx - k from the half spectra A, B of rows t0, t0 + 1
__device__ __forceinline__ void retangle(double2 *line, int k, int Nx, double2 A, double2 B) {
    if (k == 0 || 2 * k == Nx) A.y = B.y = 0.0;
    line[fft_at(k)] = make_double2(A.x - B.y, A.y + B.x);
    if (k > 0 && 2 * k != Nx) line[fft_at(Nx - k)] = make_double2(A.x + B.y, B.x - A.y);
}

// ---------------------------------------------------------------------------
// pass 1: Philox field + forward row FFTs (two rows per complex transform)
// grid: (ceil(Nt / (2*lpb)), nRep)
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(kLineThreads) YCN_FOUR_WAVES
k_noise_rows_fwd(const double *__restrict__ xi, const uint64_t *__restrict__ seeds, uint64_t step,
                 double2 *__restrict__ spec, int Nt, int Nx, int H, int nk, int lpb, FftPlan P, const StepCtl *ctl) {
    extern __shared__ double2 lds[];
    if (ctl) {   // an enqueued step: counter from the control block, nothing while halted
        if (ctl->halt) return;
        step = ctl->step;
    }
    const int row = fft_row(Nx);
    double2 *a = lds, *b = lds + lpb * row;
    const int rep = blockIdx.y;
    const int pair0 = blockIdx.x * lpb;
    load_rows(a, xi ? xi + (size_t)rep * Nt * Nx : nullptr, seeds[rep], step, pair0, lpb, Nt, Nx);
    __syncthreads();
    const double2 *res = lds_fft<false>(a, b, lpb, P);
    double2 *out = spec + (size_t)rep * Nt * H;
    const float inv = 1.0f / (float)nk;
    for (int w = threadIdx.x; w < lpb * nk; w += blockDim.x) {
        const int l = fast_div(w, inv), k = w - l * nk;
        const int t0 = 2 * (pair0 + l);
        if (t0 >= Nt) continue;
        double2 A, B;
        untangle(res + l * row, k, Nx, A, B);
        out[(size_t)t0 * H + k] = A;
        if (t0 + 1 < Nt) out[(size_t)(t0 + 1) * H + k] = B;
    }
}

// ---------------------------------------------------------------------------
// pass 2: column FFT along t, mask, inverse FFT along t (in place)
// grid: (ceil(nk / lpb), nRep).  Neighbouring column groups share the cache lines of their
// rows, so blocks are handed to the 8 XCDs in contiguous bands of groups.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(kLineThreads) YCN_FOUR_WAVES
k_noise_cols(double2 *__restrict__ spec, const int *__restrict__ kmax, int nk, double invV, int Nt, int H, int lpb,
             FftPlan P, const StepCtl *ctl) {
    extern __shared__ double2 lds[];
    if (ctl && ctl->halt) return;
    const int row = fft_row(Nt);
    double2 *a = lds, *b = lds + lpb * row;
    const int rep = blockIdx.y, nb = gridDim.x;
    const int band = (nb + 7) / 8, full = nb % 8 == 0 ? 8 : nb % 8;   // XCDs 0 .. full - 1 hold `band` groups
    const int xcd = blockIdx.x % 8;
    const int g = xcd * band - max(0, xcd - full) + (int)blockIdx.x / 8;
    const int k0 = g * lpb;
    const int nl = min(lpb, nk - k0);
    double2 *s = spec + (size_t)rep * Nt * H;
    const float inv = 1.0f / (float)lpb;
    batched<8, double2>(
        lpb * Nt,
        [&](int w) {
            const int t = fast_div(w, inv), l = w - t * lpb;
            return l < nl ? s[(size_t)t * H + k0 + l] : make_double2(0.0, 0.0);
        },
        [&](int w, double2 v) {
            const int t = fast_div(w, inv), l = w - t * lpb;
            a[l * row + fft_at(t)] = v;
        });
    __syncthreads();
    double2 *res = lds_fft<false>(a, b, lpb, P);
    double2 *oth = (res == a) ? b : a;
    batched<8, int>(
        lpb * Nt, [&](int w) { return kmax[fast_div(w, inv)]; },
        [&](int w, int km) {
            const int kt = fast_div(w, inv), l = w - kt * lpb;
            const int at = l * row + fft_at(kt);
            res[at] = cscl(k0 + l <= km ? invV : 0.0, res[at]);
        });
    __syncthreads();
    const double2 *fin = lds_fft<true>(res, oth, lpb, P);
    for (int w = threadIdx.x; w < lpb * Nt; w += blockDim.x) {
        const int t = fast_div(w, inv), l = w - t * lpb;
        if (l < nl) s[(size_t)t * H + k0 + l] = fin[l * row + fft_at(t)];
    }
}

// ---------------------------------------------------------------------------
// pass 3: inverse row FFTs (C2R), two rows per complex transform
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(kLineThreads) YCN_FOUR_WAVES
k_noise_rows_inv(const double2 *__restrict__ spec, double *__restrict__ noise, int Nt, int Nx, int H, int nk, int lpb,
                 FftPlan P, const StepCtl *ctl) {
    extern __shared__ double2 lds[];
    if (ctl && ctl->halt) return;
    const int row = fft_row(Nx);
    double2 *a = lds, *b = lds + lpb * row;
    const int rep = blockIdx.y;
    const int pair0 = blockIdx.x * lpb;
    const double2 *s = spec + (size_t)rep * Nt * H;
    const float inv = 1.0f / (float)H;
    batched<4, RowPair>(
        lpb * H,
        [&](int w) {
            const int l = fast_div(w, inv), k = w - l * H;
            const int t0 = 2 * (pair0 + l);
            RowPair v = {make_double2(0.0, 0.0), make_double2(0.0, 0.0)};
            if (t0 < Nt && k < nk) {
                v.A = s[(size_t)t0 * H + k];
                if (t0 + 1 < Nt) v.B = s[(size_t)(t0 + 1) * H + k];
            }
            return v;
        },
        [&](int w, RowPair v) {
            const int l = fast_div(w, inv), k = w - l * H;
            retangle(a + l * row, k, Nx, v.A, v.B);
        });
    __syncthreads();
    const double2 *res = lds_fft<true>(a, b, lpb, P);
    double *o = noise + (size_t)rep * Nt * Nx;
    const float invX = 1.0f / (float)Nx;
    for (int w = threadIdx.x; w < lpb * Nx; w += blockDim.x) {
        const int l = fast_div(w, invX), x = w - l * Nx;
        const int t0 = 2 * (pair0 + l);
        if (t0 >= Nt) continue;
        const double2 z = res[l * row + fft_at(x)];
        o[(size_t)t0 * Nx + x] = z.x;
        if (t0 + 1 < Nt) o[(size_t)(t0 + 1) * Nx + x] = z.y;
    }
}

// ---------------------------------------------------------------------------
// the three passes of a small lattice by one block per replica and step (step + blockIdx.y, the
// fields one after the other), the spectrum in LDS (buffers of `cap` entries): the same arithmetic
// in one launch
// ---------------------------------------------------------------------------
constexpr int kOneThreads = 512;
constexpr int kOneLdsBytes = 81920;
// TW: with the twiddle tables behind the buffers, one entry per thread
template <bool TW>
__global__ void __launch_bounds__(kOneThreads) YCN_FOUR_WAVES
k_noise_one(const double *__restrict__ xi, const uint64_t *__restrict__ seeds, uint64_t step,
            const int *__restrict__ kmax, int nk, double invV, double *__restrict__ noise, int Nt, int Nx, int cap,
            FftPlan PX, FftPlan PT, const StepCtl *ctl) {
    extern __shared__ double2 lds[];
    if (ctl) {
        if (ctl->halt) return;
        step = ctl->step;
    }
    step += blockIdx.y;
    noise += (size_t)blockIdx.y * gridDim.x * Nt * Nx;
    const int rep = blockIdx.x, np = (Nt + 1) / 2, H = Nx / 2 + 1, rowX = fft_row(Nx), rowT = fft_row(Nt);
    double2 *a = lds, *b = lds + cap;
    const double2 *twX = PX.tw, *twT = PT.tw;
    double2 wx, wt;
    if constexpr (TW) {   // requested here, in LDS once the field is made
        if ((int)threadIdx.x < Nx) wx = PX.tw[threadIdx.x];
        if ((int)threadIdx.x < Nt) wt = PT.tw[threadIdx.x];
    }
    load_rows(a, xi ? xi + (size_t)rep * Nt * Nx : nullptr, seeds[rep], step, 0, np, Nt, Nx);
    if constexpr (TW) {
        double2 *const w = lds + 2 * cap;
        if ((int)threadIdx.x < Nx) w[threadIdx.x] = wx;
        if ((int)threadIdx.x < Nt) w[Nx + threadIdx.x] = wt;
        twX = w;
        twT = w + Nx;
    }
    __syncthreads();
    double2 *res = lds_fft<false>(a, b, np, PX, twX);
    double2 *oth = (res == a) ? b : a;
    const float invK = 1.0f / (float)nk, invT = 1.0f / (float)Nt, invH = 1.0f / (float)H, invX = 1.0f / (float)Nx;
    for (int w = threadIdx.x; w < np * nk; w += blockDim.x) {
        const int l = fast_div(w, invK), k = w - l * nk;
        double2 A, B;
        untangle(res + l * rowX, k, Nx, A, B);
        oth[k * rowT + fft_at(2 * l)] = A;
        if (2 * l + 1 < Nt) oth[k * rowT + fft_at(2 * l + 1)] = B;
    }
    __syncthreads();
    double2 *col = lds_fft<false>(oth, res, nk, PT, twT);
    oth = (col == oth) ? res : oth;
    batched<4, int>(
        nk * Nt, [&](int w) { return kmax[w - fast_div(w, invT) * Nt]; },
        [&](int w, int km) {
            const int k = fast_div(w, invT), kt = w - k * Nt;
            const int at = k * rowT + fft_at(kt);
            col[at] = cscl((k <= km) ? invV : 0.0, col[at]);
        });
    __syncthreads();
    double2 *fin = lds_fft<true>(col, oth, nk, PT, twT);
    oth = (fin == a) ? b : a;
    for (int w = threadIdx.x; w < np * H; w += blockDim.x) {
        const int l = fast_div(w, invH), k = w - l * H;
        double2 A = make_double2(0.0, 0.0), B = A;
        if (k < nk) {
            A = fin[k * rowT + fft_at(2 * l)];
            if (2 * l + 1 < Nt) B = fin[k * rowT + fft_at(2 * l + 1)];
        }
        retangle(oth + l * rowX, k, Nx, A, B);
    }
    __syncthreads();
    const double2 *out = lds_fft<true>(oth, fin, np, PX, twX);
    double *o = noise + (size_t)rep * Nt * Nx;
    for (int w = threadIdx.x; w < np * Nx; w += blockDim.x) {
        const int l = fast_div(w, invX), x = w - l * Nx;
        const double2 z = out[l * rowX + fft_at(x)];
        o[(size_t)(2 * l) * Nx + x] = z.x;
        if (2 * l + 1 < Nt) o[(size_t)(2 * l + 1) * Nx + x] = z.y;
    }
}

// twiddle table tw[e] = exp(-2 pi i e / n), e < n (both entry points build it this way,
// so their transforms agree bit for bit)
__device__ __forceinline__ double2 twiddle(int e, int n) {
    double s, c;
    sincospi(-2.0 * (double)e / (double)n, &s, &c);
    return make_double2(c, s);
}
__global__ void __launch_bounds__(kFftThreads) k_twiddles(double2 *__restrict__ tw, int n) {
    const int e = blockIdx.x * kFftThreads + threadIdx.x;
    if (e < n) tw[e] = twiddle(e, n);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// Passes of a transform of length n, its power of two first: radix 8 with one or two of radix 4, or
// radix 4 alone for lines of up to 32, where a radix-8 butterfly leaves most lanes idle (256 x 256:
// 26.0 us a field with radix 4 alone, 24.8 so, 35.7 with radix 16; 512 x 512 31.2, 27.8, 28.3;
// 64 x 64 23.3, 20.3, 20.4).  Then 3, 5, 7 and the other odd primes (direct DFTs).  false if more
// than kMaxFactors are needed.
static bool factor_plan(int n, FftPlan &P) {
    P.n = n;
    P.nf = 0;
    int m = n, e = 0, Ns = 1;
    while (m % 2 == 0) {
        m /= 2;
        ++e;
    }
    auto put = [&](int r) {
        if (P.nf < kMaxFactors) {
            FftPass &F = P.pass[P.nf];
            F.R = r;
            F.nb = n / r;
            F.Ns = Ns;
            F.tstride = F.nb / Ns;
            F.invNb = 1.0f / (float)F.nb;
            F.invNs = 1.0f / (float)Ns;
        }
        ++P.nf;
        Ns *= r;
    };
    if (n <= 32 || e <= 2) {
        for (; e >= 2; e -= 2) put(4);
        if (e) put(2);
    } else {
        int fours = e % 3 == 1 ? 2 : e % 3 == 2 ? 1 : 0;   // 2^e = 8 ... 8 x 4 ... 4
        for (e -= 2 * fours; e > 0; e -= 3) put(8);
        for (; fours > 0; --fours) put(4);
    }
    for (int q = 3; m > 1; q += 2)
        while (m % q == 0) {
            put(q);
            m /= q;
        }
    return P.nf <= kMaxFactors;
}

static int make_plan(Ctx &c, int n, FftPlan &P) {
    if (!factor_plan(n, P)) { c.err = "FFT length has too many factors"; return YCN_ERR_UNSUPPORTED; }
    double2 *d = nullptr;
    YCN_HIP(hipMalloc(&d, sizeof(double2) * n));
    hipLaunchKernelGGL(k_twiddles, dim3((n + kFftThreads - 1) / kFftThreads), dim3(kFftThreads), 0, c.stream, d, n);
    YCN_HIP(hipGetLastError());
    P.tw = d;
    return YCN_OK;
}

// GlobalCoordinateToMomentumSquared (colouredNoise.cpp:16-29) and the mask build
// (:138-145), evaluated on the host in the same IEEE order (no contraction), reduced
// to kmax[kt] = largest kept kx of row kt (the kept set of a row is a prefix because
// p_x^2 grows with kx).
#pragma clang fp contract(off)
static double momentum_squared(int Nt, int Nx, int ct, int cx) {
    const int sizes[2] = {Nt, Nx}, coo[2] = {ct, cx};
    double msq = 0.0, sgn = 1.0;
    if (coo[1] > (int)std::floor(Nx / 2)) sgn = -1.0;
    for (int n = 0; n < 2; ++n) {
        const int full = sizes[n];
        const double tmp = (coo[n] <= (int)std::floor(full / 2) ? coo[n] : coo[n] - full) * 2.0 * M_PI / full;
        msq += tmp * tmp;
    }
    return msq * sgn;
}

// (s sqrt(d) pi)^2, the cutoff of colouredNoise.cpp:138-145 in its arithmetic order
static double cut_squared(double cutFraction) {
    const double cut = std::sqrt(2.0) * M_PI * cutFraction;
    return cut * cut;
}

static int build_mask(Ctx &c, std::vector<int> &kmax) {
    const int Nt = c.p.Nt, Nx = c.p.Nx, H = c.H;
    const double cutSq = cut_squared(c.p.cutFraction);
    kmax.assign(Nt, -1);
    for (int t = 0; t < Nt; ++t) {
        bool prefix = true;
        for (int k = 0; k < H; ++k) {
            const double m = momentum_squared(Nt, Nx, t, k);
            const bool keep = (m >= 0) && (m <= cutSq);
            if (keep) {
                if (kmax[t] != k - 1) prefix = false;
                kmax[t] = k;
            }
        }
        if (!prefix) { c.err = "coloured-noise mask row is not a prefix"; return YCN_ERR_UNSUPPORTED; }
    }
    return YCN_OK;
}
#pragma clang fp contract(on)

// Lines per block of a pass over `lines` lines of length n (all replicas): as few as give
// 512 blocks (two per CU), within the LDS of a block, and at least `least` where the lattice
// has them (columns: two neighbouring ones, 32 bytes of each row).
static int lines_per_block(int n, int lines, int least) {
    const int most = std::max(1, kFftLdsBytes / (2 * (int)sizeof(double2) * fft_row(n)));
    return std::min(most, std::max(least, lines / 512));
}
// threads of such a block: two points each, so that the generation, the loads and the stores are
// short chains; the radix-8 butterflies then leave half of the lanes idle
static int fft_threads(int points) {
    return std::min(kLineThreads, std::max(kWave, (points / 2 + kWave - 1) / kWave * kWave));
}
// entries of one LDS buffer of the one-block form
static int one_block_entries(int Nt, int Nx, int nk) {
    return std::max((Nt + 1) / 2 * fft_row(Nx), nk * fft_row(Nt));
}

int noise_init(Ctx &c) {
    const int Nt = c.p.Nt, Nx = c.p.Nx;
    if ((size_t)2 * sizeof(double2) * fft_row(std::max(Nt, Nx)) > (size_t)kFftLdsBytes) {
        c.err = "lattice extent too large for the LDS FFT (max 2048)";
        return YCN_ERR_UNSUPPORTED;
    }
    int rc = make_plan(c, Nx, c.planX);
    if (rc) return rc;
    rc = make_plan(c, Nt, c.planT);
    if (rc) return rc;
    std::vector<int> km;
    rc = build_mask(c, km);
    if (rc) return rc;
    c.kmaxAll = -1;
    for (int v : km) c.kmaxAll = std::max(c.kmaxAll, v);
    YCN_HIP(hipMalloc(&c.kmax, sizeof(int) * Nt));
    YCN_HIP(hipMemcpy(c.kmax, km.data(), sizeof(int) * Nt, hipMemcpyHostToDevice));
    YCN_HIP(hipMalloc(&c.spec, sizeof(double2) * (size_t)c.nRep * Nt * c.H));
    return YCN_OK;
}

void noise_free(Ctx &c) {
    if (c.planX.tw) (void)hipFree((void *)c.planX.tw);
    if (c.planT.tw) (void)hipFree((void *)c.planT.tw);
    if (c.kmax) (void)hipFree(c.kmax);
    if (c.spec) (void)hipFree(c.spec);
    c.planX.tw = c.planT.tw = nullptr;
    c.kmax = nullptr;
    c.spec = nullptr;
}

int noise_generate(Ctx &c, uint64_t step, const double *xi_dev, double *out_dev) {
    return noise_generate_on(c, c.stream, step, xi_dev, out_dev);
}

// the three noise kernels on stream s over explicit buffers (a context's, or the
// scratch array of the allocation-free entry point); prof (optional) brackets the
// column pass for a context's kernel timing
static int launch_noise(hipStream_t s, int Nt, int Nx, int nRep, const double *xi_dev, const uint64_t *seeds,
                        uint64_t step, double2 *spec, const int *kmax, int kmaxAll, const FftPlan &planX,
                        const FftPlan &planT, double *out_dev, Ctx *prof, const StepCtl *ctl = nullptr,
                        int nsteps = 1) {
    const int H = Nx / 2 + 1, nk = kmaxAll + 1;   // columns up to the cutoff
    const double invV = 1.0 / ((double)Nt * (double)Nx);
    const int npairs = (Nt + 1) / 2;
    // One block per replica where the half spectrum fits it.  Three launches take about 5 us
    // each on a small lattice, one block about 8 us for all of a 64 x 64 one; its time grows
    // with the lattice while theirs does not.
    const int cap = one_block_entries(Nt, Nx, std::max(nk, 1));
    const size_t shOne = (size_t)2 * cap * sizeof(double2);
    if (shOne <= (size_t)kOneLdsBytes) {
        if (prof) prof_before(*prof, PK_NOISE_COLS, 40.0 * (double)nRep * Nt * Nx);
        // its twiddles in LDS too, where they leave room for a second block (a pass then waits for
        // LDS instead of the caches: 12 of 45 x 50 19.6 -> 18.5 us, 5 of 64 x 64 20.6 -> 19.4)
        const size_t shTw = shOne + (size_t)(Nx + Nt) * sizeof(double2);
        const bool tw = shTw <= (size_t)kOneLdsBytes && std::max(Nx, Nt) <= kOneThreads;
        hipLaunchKernelGGL(tw ? &k_noise_one<true> : &k_noise_one<false>, dim3(nRep, nsteps), dim3(kOneThreads),
                           tw ? shTw : shOne, s, xi_dev, seeds, step, kmax, nk, invV, out_dev, Nt, Nx, cap, planX,
                           planT, ctl);
        if (prof) prof_after(*prof, PK_NOISE_COLS);
        return hipGetLastError() == hipSuccess ? YCN_OK : YCN_ERR_HIP;
    }
    if (nsteps > 1) {
        for (int i = 0; i < nsteps; ++i)
            if (launch_noise(s, Nt, Nx, nRep, xi_dev, seeds, step + i, spec, kmax, kmaxAll, planX, planT,
                             out_dev + (size_t)i * nRep * Nt * Nx, prof, ctl))
                return YCN_ERR_HIP;
        return YCN_OK;
    }
    const int lx = lines_per_block(Nx, npairs * nRep, 1), lt = lines_per_block(Nt, nk * nRep, 2);
    dim3 g1((npairs + lx - 1) / lx, nRep), g2((nk + lt - 1) / lt, nRep);
    const dim3 b1(fft_threads(lx * Nx)), b2(fft_threads(lt * Nt));
    const size_t sh1 = (size_t)2 * lx * fft_row(Nx) * sizeof(double2);
    const size_t sh2 = (size_t)2 * lt * fft_row(Nt) * sizeof(double2);
    hipLaunchKernelGGL(k_noise_rows_fwd, g1, b1, sh1, s, xi_dev, seeds, step, spec, Nt, Nx, H, nk, lx, planX, ctl);
    if (nk > 0) {
        if (prof) prof_before(*prof, PK_NOISE_COLS, 32.0 * (double)nRep * Nt * nk);
        hipLaunchKernelGGL(k_noise_cols, g2, b2, sh2, s, spec, kmax, nk, invV, Nt, H, lt, planT, ctl);
        if (prof) prof_after(*prof, PK_NOISE_COLS);
    }
    hipLaunchKernelGGL(k_noise_rows_inv, g1, b1, sh1, s, (const double2 *)spec, out_dev, Nt, Nx, H, nk, lx, planX, ctl);
    return hipGetLastError() == hipSuccess ? YCN_OK : YCN_ERR_HIP;
}

int noise_generate_on(Ctx &c, hipStream_t s, uint64_t step, const double *xi_dev, double *out_dev) {
    const int rc = launch_noise(s, c.p.Nt, c.p.Nx, c.nRep, xi_dev, (const uint64_t *)c.seed_d, step, c.spec,
                                (const int *)c.kmax, c.kmaxAll, c.planX, c.planT, out_dev, &c);
    if (rc) c.err = "coloured-noise kernel launch failed";
    return rc;
}

// the fields of nsteps consecutive steps, one after the other
int noise_generate_steps(Ctx &c, uint64_t step, int nsteps, double *out_dev) {
    const int rc = launch_noise(c.stream, c.p.Nt, c.p.Nx, c.nRep, nullptr, (const uint64_t *)c.seed_d, step, c.spec,
                                (const int *)c.kmax, c.kmaxAll, c.planX, c.planT, out_dev, &c, nullptr, nsteps);
    if (rc) c.err = "coloured-noise kernel launch failed";
    return rc;
}

int noise_generate_ctl(Ctx &c, hipStream_t s, const StepCtl *ctl, double *out_dev) {
    const int rc = launch_noise(s, c.p.Nt, c.p.Nx, c.nRep, nullptr, (const uint64_t *)c.seed_d, 0, c.spec,
                                (const int *)c.kmax, c.kmaxAll, c.planX, c.planT, out_dev, nullptr, ctl);
    if (rc) c.err = "coloured-noise kernel launch failed";
    return rc;
}

// ===========================================================================
// Coloured noise without a context and without allocations
// (ycn_coloured_noise_noalloc, for callers that cannot allocate device memory).
// Its scratch -- the half spectrum, the two twiddle tables, the mask rows and the
// replica seeds -- lives in one file-scope device array of fixed size.  Each device
// holds its own copy at its own address, looked up once per device with
// hipGetSymbolAddress; host code uses only that address, never the array's name.
// Every call on a device shares the array: calls that overlap on one device race.
// Nothing in it needs clearing: each call writes every entry it reads.
// ===========================================================================
constexpr size_t kNaSpec = (size_t)1024 * 513;   // half-spectrum entries (double2): one 1024^2 lattice
constexpr int kNaMaxN = 2048;                     // largest extent (the LDS FFT's limit)
constexpr int kNaMaxRep = 64;                     // replicas (their seeds pass by value)
constexpr int kNaMaxDevices = 64;
constexpr size_t kNaOffTwX = kNaSpec * sizeof(double2);
constexpr size_t kNaOffTwT = kNaOffTwX + kNaMaxN * sizeof(double2);
constexpr size_t kNaOffKmax = kNaOffTwT + kNaMaxN * sizeof(double2);
constexpr size_t kNaOffSeed = kNaOffKmax + kNaMaxN * sizeof(int);
constexpr size_t kNaBytes = kNaOffSeed + kNaMaxRep * sizeof(uint64_t);   // 8 479 232 B

static __device__ __align__(256) unsigned char scratch[kNaBytes];

static void *g_naScratch[kNaMaxDevices];   // the array's address on each device
static std::mutex g_naMutex;
static thread_local const char *g_naErr = nullptr;

// address of `scratch` on device dev, which must be current; looked up once per device
static int na_scratch(int dev, unsigned char **out) {
    std::lock_guard<std::mutex> lock(g_naMutex);
    if (!g_naScratch[dev]) {
        void *ptr = nullptr;
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess || !ptr) return YCN_ERR_HIP;
        g_naScratch[dev] = ptr;
    }
    *out = (unsigned char *)g_naScratch[dev];
    return YCN_OK;
}

int noise_noalloc_setup(int dev) {
    unsigned char *p = nullptr;
    if (dev < 0 || dev >= kNaMaxDevices) return YCN_ERR_INVALID;
    return na_scratch(dev, &p);
}

const char *noise_noalloc_error() { return g_naErr; }

struct NaSeeds {
    uint64_t v[kNaMaxRep];
};

// kmax[kt] of the mask on the device, in the host's IEEE order (momentum_squared, no
// contraction; correctly rounded double multiply, divide and add), so both entry points
// keep the same modes.  The kept set of a row is a prefix (checked on the host path).
#pragma clang fp contract(off)
__device__ double na_coord_sq(int c, int n) {
    const double k = (double)(c <= n / 2 ? c : c - n);
    const double t = __ddiv_rn(__dmul_rn(__dmul_rn(k, 2.0), M_PI), (double)n);
    return __dmul_rn(t, t);
}
// rows keep a prefix of their columns (the rounded momentum grows with k): its end by
// bisection
__device__ int na_kmax(int kt, int Nt, int Nx, int H, double cutSq) {
    const double mt = __dadd_rn(0.0, na_coord_sq(kt, Nt));
    int lo = -1, hi = H;   // kept up to lo, cut from hi on
    while (hi - lo > 1) {
        const int k = (lo + hi) / 2;
        const double m = __dadd_rn(mt, na_coord_sq(k, Nx));
        if (m >= 0.0 && m <= cutSq)
            lo = k;
        else
            hi = k;
    }
    return lo;
}
#pragma clang fp contract(on)

// everything a call reads besides its arguments, in one launch: block row 0 fills the x
// twiddles, row 1 the t twiddles, row 2 the mask rows and the seeds (one launch of about 5 us
// for the 56 us that a serial search per mask row and four launches took at 1024 x 1024)
__global__ void __launch_bounds__(kFftThreads)
k_na_setup(NaSeeds s, int nRep, uint64_t *__restrict__ seeds, double2 *__restrict__ twX, double2 *__restrict__ twT,
           int *__restrict__ kmax, int Nt, int Nx, int H, double cutSq) {
    const int e = blockIdx.x * kFftThreads + threadIdx.x;
    if (blockIdx.y == 0) {
        if (e < Nx) twX[e] = twiddle(e, Nx);
    } else if (blockIdx.y == 1) {
        if (e < Nt) twT[e] = twiddle(e, Nt);
    } else {
        if (e < Nt) kmax[e] = na_kmax(e, Nt, Nx, H, cutSq);
        if (e < nRep) seeds[e] = s.v[e];
    }
}

// largest kept kx over all rows: row kt = 0 (p_t = 0) keeps the most, since adding
// p_t^2 >= 0 and rounding cannot lower the momentum
static int na_kmax_all(int Nt, int Nx, double cutSq) {
    int km = -1;
    for (int k = 0; k < Nx / 2 + 1; ++k) {
        const double m = momentum_squared(Nt, Nx, 0, k);
        if (!(m >= 0 && m <= cutSq)) break;
        km = k;
    }
    return km;
}

static int na_fail(const char *msg, int code) {
    g_naErr = msg;
    return code;
}

static int na_run(const ycn_params *p, const uint64_t *seeds, uint64_t step, double *noise, hipStream_t s) {
    const int Nt = p->Nt, Nx = p->Nx, nRep = p->nReplicas, H = Nx / 2 + 1;
    FftPlan pX{}, pT{};
    if (!factor_plan(Nx, pX) || !factor_plan(Nt, pT)) return na_fail("FFT length has too many factors", YCN_ERR_UNSUPPORTED);
    unsigned char *base = nullptr;
    if (na_scratch(p->device, &base)) return na_fail("hipGetSymbolAddress of the scratch array failed", YCN_ERR_HIP);
    double2 *spec = (double2 *)base;
    double2 *twX = (double2 *)(base + kNaOffTwX), *twT = (double2 *)(base + kNaOffTwT);
    int *kmax = (int *)(base + kNaOffKmax);
    uint64_t *seed_d = (uint64_t *)(base + kNaOffSeed);
    NaSeeds sd{};
    for (int i = 0; i < nRep; ++i) sd.v[i] = seeds ? seeds[i] : p->seed;
    const double cutSq = cut_squared(p->cutFraction);
    const int blocks = (std::max({Nx, Nt, nRep}) + kFftThreads - 1) / kFftThreads;
    hipLaunchKernelGGL(k_na_setup, dim3(blocks, 3), dim3(kFftThreads), 0, s, sd, nRep, seed_d, twX, twT, kmax, Nt, Nx, H,
                       cutSq);
    pX.tw = twX;
    pT.tw = twT;
    if (launch_noise(s, Nt, Nx, nRep, nullptr, seed_d, step, spec, kmax, na_kmax_all(Nt, Nx, cutSq), pX, pT, noise,
                     nullptr))
        return na_fail("coloured-noise kernel launch failed", YCN_ERR_HIP);
    return YCN_OK;
}

}  // namespace ycn

extern "C" int ycn_coloured_noise_noalloc(const ycn_params *p, const uint64_t *seeds, uint64_t step, double *noise,
                                          void *stream) {
    using namespace ycn;
    if (!p || !noise) return na_fail("ycn_coloured_noise_noalloc: null params or output", YCN_ERR_INVALID);
    if (p->Nt < 2 || p->Nx < 2 || p->nReplicas < 1)
        return na_fail("ycn_coloured_noise_noalloc: needs Nt, Nx >= 2 and nReplicas >= 1", YCN_ERR_INVALID);
    if (p->Nt > kNaMaxN || p->Nx > kNaMaxN)
        return na_fail("ycn_coloured_noise_noalloc: Nt and Nx are limited to 2048", YCN_ERR_INVALID);
    if (p->nReplicas > kNaMaxRep)
        return na_fail("ycn_coloured_noise_noalloc: nReplicas is limited to 64", YCN_ERR_INVALID);
    if ((size_t)p->nReplicas * p->Nt * (p->Nx / 2 + 1) > kNaSpec)
        return na_fail("ycn_coloured_noise_noalloc: nReplicas * Nt * (Nx/2 + 1) exceeds the scratch capacity "
                       "1024 * 513 (one 1024^2 lattice)",
                       YCN_ERR_INVALID);
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev <= 0)
        return na_fail("ycn_coloured_noise_noalloc: no HIP device", YCN_ERR_NO_DEVICE);
    if (p->device < 0 || p->device >= ndev || p->device >= kNaMaxDevices)
        return na_fail("ycn_coloured_noise_noalloc: invalid device", YCN_ERR_INVALID);
    int prev = -1;
    if (hipGetDevice(&prev) != hipSuccess) return na_fail("ycn_coloured_noise_noalloc: hipGetDevice failed", YCN_ERR_HIP);
    if (prev != p->device && hipSetDevice(p->device) != hipSuccess)
        return na_fail("ycn_coloured_noise_noalloc: hipSetDevice failed", YCN_ERR_HIP);
    const int rc = na_run(p, seeds, step, noise, (hipStream_t)stream);
    if (prev != p->device) (void)hipSetDevice(prev);
    return rc;
}
