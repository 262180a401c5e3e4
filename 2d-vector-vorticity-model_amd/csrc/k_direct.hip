// k_direct.hip -- direct solve of the cal_w system (direct.h).
//
// Three kernels: the forward row transforms, the tridiagonal systems, the
// inverse row transforms.  At 2048 x 255 they move 8 + 10 + 12 MB in 12.7, 12.7
// and 11.6 us and are bound by latency: the rows' and the twiddles' first load
// (2 to 3 us; 5.5 where each was waited for in a branch of its own, 15 us a
// kernel), four LDS round trips of 1 us, the elimination's serial chain.
#include <algorithm>
#include <cmath>
#include <complex>
#include <type_traits>
#include <vector>

#include "direct.h"
#include "micro.h"
#include "pubartop.h"

namespace vvmd {

namespace {

// ---------------------------------------------------------- row transforms
//
// One workgroup transforms two rows at once, as the real and imaginary part
// of one complex FFT in LDS; the two spectra are separated as they leave.
// The FFT is Stockham's: each stage reads its inputs N/R apart and writes
// them in order, all reads before a barrier and all writes after it, so one
// buffer is enough (8192 columns in FP64 take 135 KB).  Real and imaginary
// parts lie in separate arrays with one word of padding every 32, which makes
// the strided writes of the first stages conflict-free.

__device__ inline int pad(int i) { return i + (i >> 5); }

template <typename T>
struct Cx {
    T x, y;
};
template <typename T>
__device__ inline Cx<T> operator+(Cx<T> a, Cx<T> b) {
    return {a.x + b.x, a.y + b.y};
}
template <typename T>
__device__ inline Cx<T> operator-(Cx<T> a, Cx<T> b) {
    return {a.x - b.x, a.y - b.y};
}
template <typename T>
__device__ inline Cx<T> mul(Cx<T> a, Cx<T> b) {
    return {a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
template <typename T>
__device__ inline Cx<T> mul_mi(Cx<T> a) {  // -i a
    return {a.y, -a.x};
}

// Forward DFTs of R values in place (kernel exp(-2 pi i / R)).
template <typename T>
__device__ inline void dft2(Cx<T> &a, Cx<T> &b) {
    const Cx<T> t = a;
    a = t + b;
    b = t - b;
}
template <typename T>
__device__ inline void dft4(Cx<T> &a, Cx<T> &b, Cx<T> &c, Cx<T> &d) {
    dft2(a, c);
    dft2(b, d);
    d = mul_mi(d);
    dft2(a, b);
    dft2(c, d);
    const Cx<T> t = b;  // bit-reversed order back to natural
    b = c;
    c = t;
}

// odd R: cos and sin of 2 pi k / R, k = 1..(R-1)/2
template <int R>
struct Roots;
template <>
struct Roots<3> {
    static constexpr double c[1] = {-0.5}, s[1] = {8.66025403784438646764e-01};
};
template <>
struct Roots<5> {
    static constexpr double c[2] = {3.09016994374947424102e-01, -8.09016994374947424102e-01},
                            s[2] = {9.51056516295153572116e-01, 5.87785252292473129169e-01};
};
template <int R, typename T>
__device__ inline void dft(Cx<T> (&v)[R]) {
    if constexpr (R == 2) {
        dft2(v[0], v[1]);
    } else if constexpr (R == 4) {
        dft4(v[0], v[1], v[2], v[3]);
    } else if constexpr (R == 8) {
        constexpr T h = T(0.70710678118654752440);
        dft4(v[0], v[2], v[4], v[6]);
        dft4(v[1], v[3], v[5], v[7]);
        // odd part times exp(-2 pi i k / 8)
        const Cx<T> o0 = v[1], o1{h * (v[3].x + v[3].y), h * (v[3].y - v[3].x)}, o2 = mul_mi(v[5]),
                    o3{h * (v[7].y - v[7].x), -h * (v[7].x + v[7].y)};
        const Cx<T> e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
        v[0] = e0 + o0;
        v[1] = e1 + o1;
        v[2] = e2 + o2;
        v[3] = e3 + o3;
        v[4] = e0 - o0;
        v[5] = e1 - o1;
        v[6] = e2 - o2;
        v[7] = e3 - o3;
    } else {
        constexpr int H = (R - 1) / 2;
        Cx<T> a[H], b[H], out[R];
        out[0] = v[0];
#pragma unroll
        for (int r = 0; r < H; r++) {
            a[r] = v[r + 1] + v[R - 1 - r];
            b[r] = v[r + 1] - v[R - 1 - r];
            out[0] = out[0] + a[r];
        }
#pragma unroll
        for (int k = 1; k <= H; k++) {
            Cx<T> p = v[0], m{T(0), T(0)};  // sums with cos and with sin
#pragma unroll
            for (int r = 1; r <= H; r++) {
                const int t = (k * r) % R, u = t <= H ? t : R - t;
                const T c = T(Roots<R>::c[u - 1]), s = t <= H ? T(Roots<R>::s[u - 1]) : -T(Roots<R>::s[u - 1]);
                p.x += c * a[r - 1].x;
                p.y += c * a[r - 1].y;
                m.x += s * b[r - 1].x;
                m.y += s * b[r - 1].y;
            }
            out[k] = {p.x + m.y, p.y - m.x};      // p - i m
            out[R - k] = {p.x - m.y, p.y + m.x};  // p + i m
        }
#pragma unroll
        for (int r = 0; r < R; r++) v[r] = out[r];
    }
}

// One Stockham stage of radix R after stages of product Ns.  NB: butterflies
// a thread, ceil(8 / R) since threads >= N / 8.  tw: exp(-2 pi i r k / (Ns R))
// at (r - 1) Ns + k, so that neighbouring threads read neighbouring values.
// A thread without a butterfly repeats the last one and stores nothing: reads
// under a branch would each be waited for before the next butterfly's are
// issued (the odd radices keep the branch, as two butterflies at once spill).
template <int R, typename T>
__device__ inline void stage(T *re, T *im, int N, int Ns, const T *__restrict__ tw) {
    constexpr int NB = (8 + R - 1) / R;
    const int nb = N / R;
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));  // addresses formed here, not for every radix ahead of all stages (they spill)
    Cx<T> v[NB][R];
    int dst[NB];
#pragma unroll
    for (int t = 0; t < NB; t++) {
        const int jt = tid + t * blockDim.x, j = min(jt, nb - 1);
        if (R % 2 && jt >= nb) continue;
        const int q = int(unsigned(j) / unsigned(Ns)), k = j - q * Ns;
        dst[t] = q * Ns * R + k;
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int a = pad(j + r * nb);
            v[t][r] = {re[a], im[a]};
        }
        if (Ns > 1) {
#pragma unroll
            for (int r = 1; r < R; r++) {
                const int a = 2 * ((r - 1) * Ns + k);
                v[t][r] = mul(v[t][r], Cx<T>{tw[a], tw[a + 1]});
            }
        }
        dft<R>(v[t]);
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NB; t++) {
        if (int(tid + t * blockDim.x) < nb) {
#pragma unroll
            for (int r = 0; r < R; r++) {
                const int a = pad(dst[t] + r * Ns);
                re[a] = v[t][r].x;
                im[a] = v[t][r].y;
            }
        }
    }
    __syncthreads();
}

// A stage of any other (prime) radix: every thread forms up to 8 outputs as
// sums over their R inputs.  O(N R) a row, for columns no one picks for speed.
template <typename T>
__device__ inline void stage_any(T *re, T *im, int N, int Ns, int R, const T *tw) {
    const int nb = N / R, m = N / (Ns * R);
    T ax[8], ay[8];
    int b[8], dst[8], step[8], idx[8];
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const int e = threadIdx.x + t * blockDim.x, ee = e < N ? e : 0;
        const int r = ee / nb;
        b[t] = ee - r * nb;
        const int q = b[t] / Ns, k = b[t] - q * Ns;
        dst[t] = q * Ns * R + k + r * Ns;
        step[t] = k * m + r * nb;  // < N
        idx[t] = 0;
        ax[t] = ay[t] = T(0);
    }
    for (int s = 0; s < R; s++) {
#pragma unroll
        for (int t = 0; t < 8; t++) {
            const int a = pad(b[t] + s * nb);
            const T vx = re[a], vy = im[a], c = tw[2 * idx[t]], d = tw[2 * idx[t] + 1];
            ax[t] += vx * c - vy * d;
            ay[t] += vx * d + vy * c;
            idx[t] += step[t];
            if (idx[t] >= N) idx[t] -= N;
        }
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < 8; t++)
        if (int(threadIdx.x + t * blockDim.x) < N) {
            const int a = pad(dst[t]);
            re[a] = ax[t];
            im[a] = ay[t];
        }
    __syncthreads();
}

// The twiddles that the transform reads from LDS (RowPlan::tw): loaded with the
// rows, so that their latency is paid once and not in every stage.
template <typename T>
struct Twiddles {
    Cx<T> v[8];
    __device__ inline void load(const RowPlan &P, const T *__restrict__ tw) {
        if (P.tw == RowPlan::TW_GLOBAL) return;
        const Cx<T> *src = reinterpret_cast<const Cx<T> *>(tw) + (P.tw == RowPlan::TW_STAGES ? P.L : 0);
#pragma unroll
        for (int t = 0; t < 8; t++) v[t] = src[min(int(threadIdx.x + t * blockDim.x), P.L - 1)];
    }
    __device__ inline void store(const RowPlan &P, T *twl) const {
        if (P.tw == RowPlan::TW_GLOBAL) return;
#pragma unroll
        for (int t = 0; t < 8; t++) {
            const int i = threadIdx.x + t * blockDim.x;
            if (i < P.L) {
                twl[2 * i] = v[t].x;
                twl[2 * i + 1] = v[t].y;
            }
        }
    }
};

template <bool LDS, bool ANY, typename T>
__device__ inline void fft_stages(const RowPlan &P, T *re, T *im, const T *tw, const T *twl) {
    const int L = P.L;
    int Ns = 1;
    for (int s = 0; s < P.nst; s++) {
        const int R = P.radix[s];
        // the stages' tables follow the table of all L roots; those before
        // hold sum (R - 1) Ns = Ns - 1 values
        const T *ts = LDS ? twl + 2 * (Ns - 1) : tw + 2 * (L + Ns - 1);
        switch (R) {
            case 8: stage<8>(re, im, L, Ns, ts); break;
            case 4: stage<4>(re, im, L, Ns, ts); break;
            case 2: stage<2>(re, im, L, Ns, ts); break;
            case 3: if constexpr (ANY) stage<3>(re, im, L, Ns, ts); break;
            case 5: if constexpr (ANY) stage<5>(re, im, L, Ns, ts); break;
            default:
                if constexpr (ANY && !LDS) stage_any(re, im, L, Ns, R, P.tw == RowPlan::TW_ROOTS ? twl : tw);
        }
        Ns *= R;
    }
}

// The transform of the N values in re, im (after a barrier).
//
// CHIRP, for large prime factors: n k = (n^2 + k^2 - (k - n)^2) / 2 makes it a
// convolution with a chirp (Bluestein's algorithm), by two transforms of length
// L = 2^j >= 2 N - 1.  The values come multiplied by the chirp c_n = exp(-i pi
// n^2 / N) and padded with zeros; bhat is the transform of 1 / c over L.  The
// inverse transform is the forward one with real and imaginary parts swapped.
// 317 columns: an isolated solve 75 us, 383 with the direct sums of 317 terms.
template <bool CHIRP, typename T>
__device__ inline void fft(const RowPlan &P, T *re, T *im, const T *__restrict__ tw, const T *twl,
                           const T *__restrict__ chirp) {
    __syncthreads();
    if constexpr (!CHIRP) {
        if (P.tw == RowPlan::TW_STAGES) fft_stages<true, true>(P, re, im, tw, twl);
        else fft_stages<false, true>(P, re, im, tw, twl);
    } else {
        auto times = [&](const T *by, int n) {
            const Cx<T> *c = reinterpret_cast<const Cx<T> *>(by);
            Cx<T> v[8];
#pragma unroll
            for (int t = 0; t < 8; t++) v[t] = c[min(int(threadIdx.x + t * blockDim.x), n - 1)];
#pragma unroll
            for (int t = 0; t < 8; t++) {
                const int i = threadIdx.x + t * blockDim.x;
                if (i < n) {
                    const Cx<T> z = mul(Cx<T>{re[pad(i)], im[pad(i)]}, v[t]);
                    re[pad(i)] = z.x;
                    im[pad(i)] = z.y;
                }
            }
            __syncthreads();
        };
        for (int pass = 0; pass < 2; pass++) {
            T *a = pass ? im : re, *b = pass ? re : im;
            if (P.tw == RowPlan::TW_STAGES) fft_stages<true, false>(P, a, b, tw, twl);
            else fft_stages<false, false>(P, a, b, tw, twl);
            if (pass == 0) times(chirp + 2 * P.N, P.L);
            else times(chirp, P.N);
        }
    }
}
// The rows' values to LDS, past the last column zeros.
template <bool CHIRP, typename T, typename V>
__device__ inline void fill_rows(const RowPlan &P, T *re, T *im, const V (&va)[8], const V (&vb)[8], bool two,
                                 const T *__restrict__ chirp) {
    const Cx<T> *c = reinterpret_cast<const Cx<T> *>(chirp);
    Cx<T> cv[8];
    if constexpr (CHIRP) {
#pragma unroll
        for (int t = 0; t < 8; t++) cv[t] = c[min(int(threadIdx.x + t * blockDim.x), P.N - 1)];
    }
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const int i = threadIdx.x + t * blockDim.x;
        Cx<T> z{T(va[t]), two ? T(vb[t]) : T(0)};
        if constexpr (CHIRP) z = i < P.N ? mul(z, cv[t]) : Cx<T>{T(0), T(0)};
        if (i < (CHIRP ? P.L : P.N)) {
            re[pad(i)] = z.x;
            im[pad(i)] = z.y;
        }
    }
}

// Hartley values (Re - Im) of the two rows at frequency q, times 2 h, from the complex
// spectrum Z of row a + i row b: A(q) = (Z(q) + Z*(N-q)) / 2,
// B(q) = (Z(q) - Z*(N-q)) / 2i.
template <typename T>
__device__ inline void hartley_pair(const T *re, const T *im, int N, int q, T h, T &ha, T &hb) {
    const int a = pad(q), c = pad(q == 0 ? 0 : N - q);
    const T zr = re[a], zi = im[a], cr = re[c], ci = im[c];
    ha = h * ((zr + cr) - (zi - ci));
    hb = h * ((zi + ci) + (zr - cr));
}

// Forward: rows j, j+1 of r (RHS false), or cal_w's right-hand side
// f = -b / rhow, b = rhow^2 (zetap[i+1] - zetap[i]) dx
// (src/PoissonSolver.cpp:444-450), formed from zetap and stored (RHS true).
// Times 1/N, the inverse transform's.
// With RHS the workgroups behind the rows' do what else has to follow the
// advection: with a step one pubarTop_pt, which reads u, w and K as the solve
// finds them (alone it was a launch of 5 to 8 us), and m.nblk Kessler.
template <typename T, bool RHS, bool CHIRP>
__global__ void __launch_bounds__(1024) k_rows_fwd(RowPlan P, const T *__restrict__ tw, const T *__restrict__ chirp,
                                                   const double *__restrict__ r,
                                                   T *__restrict__ spec, Grid G, StepPtrs S, int step,
                                                   double *__restrict__ f, Micro m) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    if constexpr (RHS) {
        note_start(S.clock, CLK_SOLVE);
        if (m.nblk) note_start(S.clock, CLK_MICRO);
        const int extra = int(blockIdx.x) - (P.M + 1) / 2, first = step >= 0 ? 1 : 0;
        if (extra >= 0) {
            if (extra < first) pubartop_block(G, S, step);
            else kessler_block(G, S, m, extra - first);
            return;
        }
    }
    const double *zetap = S.fut[F_ZETA], *rhow = S.P.rhow;
    const int N = P.N, M = P.M, LN = pad(P.L - 1) + 1;
    T *re = reinterpret_cast<T *>(lds_raw), *im = re + LN, *twl = im + LN;
    const int j = 1 + 2 * blockIdx.x;
    const bool two = j + 1 <= M;
    const int j1 = two ? j + 1 : j;
    Twiddles<T> W;
    W.load(P, tw);
    // all loads in flight at once: past the last column it is read again, and
    // nothing is waited for in a branch (a guarded load was 0.7 us, eight times)
    double va[8], vb[8];
#pragma unroll
    for (int t = 0; t < 8; t++) {  // threads >= N / 8
        const int i = min(int(threadIdx.x + t * blockDim.x), N - 1);
        if constexpr (RHS) {
            va[t] = at(zetap, G, i + 2, j + 1) - at(zetap, G, i + 1, j + 1);
            vb[t] = at(zetap, G, i + 2, j1 + 1) - at(zetap, G, i + 1, j1 + 1);
        } else {
            va[t] = r[size_t(j) * N + i];
            vb[t] = r[size_t(j1) * N + i];
        }
    }
    W.store(P, twl);
    auto rhs = [&](double d, double rw) {
#pragma clang fp contract(off)
        const double b = rw * rw * d * G.dx;
        return -b / rw;
    };
    if constexpr (RHS) {
#pragma unroll
        for (int t = 0; t < 8; t++) {
            const int i = threadIdx.x + t * blockDim.x;
            va[t] = rhs(va[t], rhow[j + 1]);
            vb[t] = rhs(vb[t], rhow[j1 + 1]);
            if (i < N) {
                f[size_t(j) * N + i] = va[t];
                if (two) f[size_t(j + 1) * N + i] = vb[t];
            }
        }
    }
    fill_rows<CHIRP>(P, re, im, va, vb, two, chirp);
    fft<CHIRP>(P, re, im, tw, twl, chirp);
    const T h = T(0.5 / N);
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const int q = threadIdx.x + t * blockDim.x;
        T ha, hb;
        hartley_pair(re, im, N, min(q, N - 1), h, ha, hb);
        if (q < N) {
            spec[size_t(j - 1) * N + q] = ha;
            if (two) spec[size_t(j) * N + q] = hb;
        }
    }
}

// Inverse: x = the transform of rows j, j+1 of spec (ADD: x0 + it); with w also
// w[i][k] = x / rhow[k] and BoundaryProcess2D_westdown(w)
// (src/PoissonSolver.cpp:469-476).
template <typename T, bool ADD, bool W, bool CHIRP>
__global__ void __launch_bounds__(1024) k_rows_inv(RowPlan P, const T *__restrict__ tw, const T *__restrict__ chirp,
                                                   const T *__restrict__ spec, const double *x0, double *x, Grid G, double *__restrict__ w,
                                                   const double *__restrict__ rhow, long long *micro_clock) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int N = P.N, M = P.M, LN = pad(P.L - 1) + 1;
    T *re = reinterpret_cast<T *>(lds_raw), *im = re + LN, *twl = im + LN;
    const int j = 1 + 2 * blockIdx.x;
    const bool two = j + 1 <= M;
    const int j1 = two ? j + 1 : j;
    Twiddles<T> Tw;
    Tw.load(P, tw);
    T va[8], vb[8];
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const int i = min(int(threadIdx.x + t * blockDim.x), N - 1);
        va[t] = spec[size_t(j - 1) * N + i];
        vb[t] = spec[size_t(j1 - 1) * N + i];
    }
    Tw.store(P, twl);
    fill_rows<CHIRP>(P, re, im, va, vb, two, chirp);
    if constexpr (W) {  // the zero rows of w
        note_start(micro_clock, CLK_MICRO_END);
        for (int i = threadIdx.x; i < G.nx; i += blockDim.x) {
            if (blockIdx.x == 0) w[ix(G, i, 0)] = w[ix(G, i, 1)] = 0.;
            if (blockIdx.x == gridDim.x - 1) w[ix(G, i, G.nz - 1)] = 0.;
        }
    }
    fft<CHIRP>(P, re, im, tw, twl, chirp);
    double xa[8], xb[8];
    if constexpr (ADD) {
#pragma unroll
        for (int t = 0; t < 8; t++) {
            const int i = min(int(threadIdx.x + t * blockDim.x), N - 1);
            xa[t] = x0[size_t(j) * N + i];
            xb[t] = x0[size_t(j1) * N + i];
        }
    }
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const int q = threadIdx.x + t * blockDim.x;
        T ha, hb;
        hartley_pair(re, im, N, min(q, N - 1), T(0.5), ha, hb);
        double da = double(ha), db = double(hb), wa = 0., wb = 0.;
        if constexpr (ADD) {
            da += xa[t];
            db += xb[t];
        }
        if constexpr (W) {
            wa = da / rhow[j + 1];
            wb = db / rhow[j1 + 1];
        }
        if (q < N) {
            x[size_t(j) * N + q] = da;
            if constexpr (W) store_westdown(w, G, q + 1, j + 1, wa);
            if (two) {
                x[size_t(j + 1) * N + q] = db;
                if constexpr (W) store_westdown(w, G, q + 1, j + 2, wb);
            }
        }
    }
}

// ------------------------------------------------------ tridiagonal systems
//
// Row j (1-based) of frequency q: d_j x_j - cu_j x_{j+1} - cu_{j-1} x_{j-1} =
// F_j.  Eliminated from both ends towards row mid = (M+1)/2 at once, which
// halves the serial chain; with the pivots p and F' = F / p,
//   downwards (j < mid): z_j = F'_j + (cu_{j-1} / p_j) z_{j-1},
//   upwards   (j > mid): z_j = F'_j + (cu_j / p_j) z_{j+1},
// at mid both, x_mid = z_mid, and back x_j = z_j + (cu_j / p_j) x_{j+1} or
// z_j + (cu_{j-1} / p_j) x_{j-1}.  Only 1 / p_j is kept, formed once, for
// q = 0..N/2 (lambda_q = lambda_{N-q}).

template <typename T>
__global__ void __launch_bounds__(64) k_factor(int N, int M, const double *__restrict__ cx,
                                               const double *__restrict__ cu, T *__restrict__ di) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x, Nq = N / 2 + 1;
    if (q >= Nq) return;
    const double s = sinpi(double(q) / N), lam = 4. * s * s;
    const int mid = (M + 1) / 2;
    auto diag = [&](int j) { return cx[j] * lam + cu[j] + cu[j - 1]; };
    double top = 0., bot = 0.;  // what the rows above and below take off p_mid
    for (int j = 1; j < mid; j++) {
        const double p = diag(j) - top;
        di[size_t(j - 1) * Nq + q] = T(1. / p);
        top = cu[j] * (cu[j] / p);
    }
    for (int j = M; j > mid; j--) {
        const double p = diag(j) - bot;
        di[size_t(j - 1) * Nq + q] = T(1. / p);
        bot = cu[j - 1] * (cu[j - 1] / p);
    }
    di[size_t(mid - 1) * Nq + q] = T(1. / (diag(mid) - top - bot));
}

// Eight columns a workgroup.  Every thread scales them and forms their factors
// on the way to LDS (all loads in flight at once), in the order of the
// elimination's steps: slot s of a direction holds its s-th row, after enough
// empty slots to make the number of steps a multiple of eight.  Then 16 lanes,
// 8 columns x 2 directions, run all steps without a branch, the next eight
// steps' values in registers: one 16-byte LDS read, one multiply-add and one
// write a step, which is the serial chain that bounds the kernel (1.4 us down,
// 2 us back for 64 steps at 1024 x 127; with three reads, a multiply and a
// kept factor more 2.4 and 1.7).  An empty slot leaves z = 0, and x is not
// read after it.  At 2048 x 255: 12.7 us, 15.5 before.
// Neighbouring workgroups share a cache line of every row, and the columns q
// and N - q their pivots: an XCD gets neighbours and their mirror images.
constexpr int KC = 8, KSTEP = 8, KL = 2 * KC;
template <typename T>
struct alignas(2 * sizeof(T)) Elim {
    T z, f;  // F', then z, then x; the elimination's factor
};
template <typename T>
struct ColStep {
    Elim<T> e[KL];
    T b[KL];  // the back substitution's factor
};
template <typename T>
struct ColMid {
    T z[KC], dn[KC], up[KC];
};
struct ColSteps {
    int mid, steps, pad_dn, pad_up;
};
__host__ __device__ inline ColSteps col_steps(int M) {
    ColSteps c;
    c.mid = (M + 1) / 2 - 1;  // 0-based
    const int dn = c.mid, up = M - 1 - c.mid, n = dn > up ? dn : up;
    c.steps = ((n > 1 ? n : 1) + KSTEP - 1) / KSTEP * KSTEP;
    c.pad_dn = c.steps - dn;
    c.pad_up = c.steps - up;
    return c;
}
template <typename T>
size_t col_lds_bytes(int M) {
    return size_t(col_steps(M).steps) * sizeof(ColStep<T>) + sizeof(ColMid<T>);
}

// With Mic the workgroups behind those of the columns do the second pass of
// the microphysics that rode in k_rows_fwd.
struct NoMicro {};
struct MicroPass {
    Grid G;
    StepPtrs S;
    Negval nv;
    int nblk;
};
template <typename T, typename Mic>
__global__ void __launch_bounds__(256) k_columns(int N, int M, T *__restrict__ spec, const T *__restrict__ di,
                                                 const double *__restrict__ cu, Mic mic) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    ColStep<T> *L = reinterpret_cast<ColStep<T> *>(lds_raw);
    const ColSteps cs = col_steps(M);
    ColMid<T> &Mid = *reinterpret_cast<ColMid<T> *>(L + cs.steps);
    const int Nq = N / 2 + 1, nt = (N + KC - 1) / KC, tile = xcd_tile(nt);
    if constexpr (std::is_same<Mic, MicroPass>::value) {
        const int extra = int(blockIdx.x) - kXcds * xcd_run(nt);
        if (extra >= 0) {
            scale_block(mic.G, mic.S, mic.nv, extra, mic.nblk);
            return;
        }
    }
    if (tile >= nt) return;
    const int b = tile % 2 ? nt - 1 - tile / 2 : tile / 2;
    // columns past the last repeat it (never stored)
    const int c = threadIdx.x % KC, q = min(b * KC + c, N - 1), qq = min(q, N - q);
    const int rstep = blockDim.x / KC;
    // step and lane of row j (0-based, not mid)
    auto step = [&](int j) { return j < cs.mid ? cs.pad_dn + j : cs.pad_up + M - 1 - j; };
    auto lane = [&](int j) { return j < cs.mid ? c : KC + c; };
    for (int j0 = threadIdx.x / KC; j0 < M; j0 += 8 * rstep) {
        T vf[8], vd[8];
        double c0[8], c1[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int j = min(j0 + u * rstep, M - 1);
            vf[u] = spec[size_t(j) * N + q];
            vd[u] = di[size_t(j) * Nq + qq];
            c0[u] = cu[j];
            c1[u] = cu[j + 1];
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int j = j0 + u * rstep;
            const T z = vf[u] * vd[u], lo = T(c0[u]) * vd[u], hi = T(c1[u]) * vd[u];
            if (j < M && j != cs.mid) {
                ColStep<T> &l = L[step(j)];
                l.e[lane(j)] = {z, j < cs.mid ? lo : hi};
                l.b[lane(j)] = j < cs.mid ? hi : lo;
            } else if (j == cs.mid) {
                Mid.z[c] = z;
                Mid.dn[c] = lo;
                Mid.up[c] = hi;
            }
        }
    }
    for (int t = threadIdx.x; t < cs.pad_dn * KC; t += blockDim.x) L[t / KC].e[t % KC] = {T(0), T(0)};
    for (int t = threadIdx.x; t < cs.pad_up * KC; t += blockDim.x) L[t / KC].e[KC + t % KC] = {T(0), T(0)};
    __syncthreads();
    if (threadIdx.x < KL) {
        __builtin_amdgcn_s_setprio(3);  // the second stream's kernels share the CU
        const int l = threadIdx.x;
        ColStep<T> *p = L;
        T z = T(0);
        Elim<T> ne[KSTEP];
#pragma unroll
        for (int u = 0; u < KSTEP; u++) ne[u] = p[u].e[l];
        for (int s = 0; s < cs.steps; s += KSTEP, p += KSTEP) {
            Elim<T> e[KSTEP];
#pragma unroll
            for (int u = 0; u < KSTEP; u++) e[u] = ne[u];
            // past the last step this reads the same eight again
            const ColStep<T> *nx = s + KSTEP < cs.steps ? p + KSTEP : p;
#pragma unroll
            for (int u = 0; u < KSTEP; u++) ne[u] = nx[u].e[l];
#pragma unroll
            for (int u = 0; u < KSTEP; u++) {
                z = e[u].z + e[u].f * z;
                p[u].e[l].z = z;
            }
        }
        const bool up = l >= KC;
        const T other = __shfl_xor(z, KC, kWave);
        // the same order of terms in both directions' lanes
        const int col = l % KC;
        T x = Mid.z[col] + Mid.dn[col] * (up ? other : z) + Mid.up[col] * (up ? z : other);
        if (!up) Mid.z[col] = x;
        p -= KSTEP;
        T nz[KSTEP], nb[KSTEP];
#pragma unroll
        for (int u = 0; u < KSTEP; u++) {
            nz[u] = p[u].e[l].z;
            nb[u] = p[u].b[l];
        }
        for (int s = cs.steps; s > 0; s -= KSTEP, p -= KSTEP) {
            T vz[KSTEP], vb[KSTEP];
#pragma unroll
            for (int u = 0; u < KSTEP; u++) {
                vz[u] = nz[u];
                vb[u] = nb[u];
            }
            const ColStep<T> *nx = s > KSTEP ? p - KSTEP : p;
#pragma unroll
            for (int u = 0; u < KSTEP; u++) {
                nz[u] = nx[u].e[l].z;
                nb[u] = nx[u].b[l];
            }
#pragma unroll
            for (int u = KSTEP - 1; u >= 0; u--) {
                x = vz[u] + vb[u] * x;
                p[u].e[l].z = x;
            }
        }
    }
    __syncthreads();
    if (b * KC + c >= N) return;
    for (int j = threadIdx.x / KC; j < M; j += rstep)
        spec[size_t(j) * N + q] = j == cs.mid ? Mid.z[c] : L[step(j)].e[lane(j)].z;
}

constexpr size_t kLdsMax = 156 * 1024;  // of a CU's 160 KiB; the sums' arrays take the rest

template <typename T>
T *dalloc(size_t n) {
    void *p = nullptr;
    if (hipMalloc(&p, n * sizeof(T)) != hipSuccess) return nullptr;
    return static_cast<T *>(p);
}

// The attribute belongs to the kernel, not to this plan: always the most that
// any plan may ask for, so that no handle lowers it under another.
template <typename K>
bool allow_lds(K kernel, size_t bytes) {
    return bytes <= 64 * 1024 || hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize,
                                                     int(kLdsMax)) == hipSuccess;
}

// exp(-2 pi i k / n)
inline std::complex<long double> root(long long k, long long n) {
    const long double a = 2.0L * 3.14159265358979323846264338327950288L * (k % n) / n;
    return {std::cos(a), -std::sin(a)};
}
// in place, forward, n a power of two; w: the n roots
void host_fft(std::vector<std::complex<long double>> &v, const std::vector<std::complex<long double>> &w) {
    const size_t n = v.size();
    for (size_t i = 1, j = 0; i < n; i++) {
        size_t bit = n >> 1;
        for (; j & bit; bit >>= 1) j ^= bit;
        j ^= bit;
        if (i < j) std::swap(v[i], v[j]);
    }
    for (size_t len = 2; len <= n; len *= 2)
        for (size_t i = 0; i < n; i += len)
            for (size_t k = 0; k < len / 2; k++) {
                const auto a = v[i + k], c = v[i + k + len / 2], r = w[k * (n / len)];
                // spelled out: std::complex's product checks for infinities
                const std::complex<long double> b(c.real() * r.real() - c.imag() * r.imag(),
                                                  c.real() * r.imag() + c.imag() * r.real());
                v[i + k] = a + b;
                v[i + k + len / 2] = a - b;
            }
}

// Up to this sum of the prime factors above 5 the direct sums are used, where
// they cost no more, to 3%, than the chirp's second transform and longer rows: at
// such a tie their residual is the smaller one (28 columns 3.7e-15 against
// 4.7e-15, 1472 8.2e-15 against 9.8e-15).  A whole isolated solve with 64 rows in
// us, sums / chirp: 28 columns (sum 7) 49.6 / 48.0, 56 49.6 / 49.9, 448 54.2 /
// 60.0, 896 57.4 / 62.2, 176 (11) 56.9 / 52.8, 208 (13) 58.8 / 52.6; for more than
// 1024 columns 1792 (7) 59.2 / 72.0, 1100 (11) 62.7 / 70.6, 1216 (19) 68.6 / 70.6,
// 1472 (23) 73.2 / 71.1, 2128 (26) 92.8 / 103.9, 2401 (28) 102.0 / 104.7, 1856
// (29) 85.3 / 72.6, 1184 (37) 89.6 / 75.3, 3059 (49) 127.6 / 106.6.  Above 1024
// the lines of 2048 and 4096 columns' chirps are not told apart (3712 (29) 101.2
// / 104.7), nor below it those of 11 and 13 (704 58.8 / 61.4, 832 61.9 / 62.1).
// With sums a prime of 317 columns took 383 us, 4093 5316.
inline int max_sums(int N) { return N <= 1024 ? 10 : 28; }

}  // namespace

template <typename T>
int Direct<T>::init(int N, int M, const double *cx, const double *cu) {
    plan = RowPlan();
    plan.N = plan.L = N;
    plan.M = M;
    int n = N;
    auto take = [&](int r) {
        while (n % r == 0 && plan.nst < kMaxStages) {
            plan.radix[plan.nst++] = r;
            n /= r;
        }
    };
    for (int r : {8, 4, 2, 3, 5}) take(r);
    const int small = plan.nst;
    int sums = 0;
    for (int r = 7; n > 1 && plan.nst < kMaxStages; r += 2) {
        if (r * r > n) r = n;
        take(r);
    }
    for (int s = small; s < plan.nst; s++) sums += plan.radix[s];
    if (n != 1 || N > 8192) return VVM_ERR_SIZE;
    if (sums > max_sums(N) && 2 * N - 1 <= 8192) {
        plan.chirp = 1;
        plan.L = 1;
        while (plan.L < 2 * N - 1) plan.L *= 2;
        plan.nst = 0;
        n = plan.L;
        for (int r : {8, 4, 2}) take(r);
    }
    const int L = plan.L;
    plan.threads = std::min(1024, std::max(64, ((L + 7) / 8 + 63) / 64 * 64));
    const size_t LN = size_t(L - 1) + size_t((L - 1) >> 5) + 1;
    row_lds = 2 * LN * sizeof(T);
    if (row_lds + 2 * size_t(L) * sizeof(T) <= kLdsMax) {
        plan.tw = sums && !plan.chirp ? RowPlan::TW_ROOTS : RowPlan::TW_STAGES;
        row_lds += 2 * size_t(L) * sizeof(T);
    }
    col_lds = col_lds_bytes<T>(M);
    if (row_lds > kLdsMax || col_lds > kLdsMax) return VVM_ERR_SIZE;
    bool ok = allow_lds(k_columns<T, NoMicro>, col_lds) && allow_lds(k_columns<T, MicroPass>, col_lds);
    auto allow_rows = [&](auto chirp) {
        constexpr bool C = decltype(chirp)::value;
        ok = ok && allow_lds(k_rows_fwd<T, false, C>, row_lds) && allow_lds(k_rows_fwd<T, true, C>, row_lds) &&
             allow_lds(k_rows_inv<T, false, false, C>, row_lds) && allow_lds(k_rows_inv<T, true, false, C>, row_lds) &&
             allow_lds(k_rows_inv<T, false, true, C>, row_lds) && allow_lds(k_rows_inv<T, true, true, C>, row_lds);
    };
    if (plan.chirp) allow_rows(std::true_type());
    else allow_rows(std::false_type());
    if (!ok) return VVM_ERR_HIP;
    const size_t Nq = size_t(N) / 2 + 1;
    tw = dalloc<T>(4 * size_t(L));
    if (plan.chirp) chirp = dalloc<T>(2 * size_t(N + L));
    di = dalloc<T>(Nq * M);
    spec = dalloc<T>(size_t(N) * M);
    if (!tw || !di || !spec || (plan.chirp && !chirp)) {
        destroy();
        return VVM_ERR_NOMEM;
    }
    std::vector<T> t(4 * size_t(L), T(0));
    std::vector<std::complex<long double>> roots(L);
    for (int k = 0; k < L; k++) {
        roots[k] = root(k, L);
        t[2 * k] = T(roots[k].real());
        t[2 * k + 1] = T(roots[k].imag());
    }
    // the stages' twiddles, picked from those (r k < Ns R, so r k L / (Ns R) < L)
    for (int s = 0, Ns = 1; s < plan.nst; Ns *= plan.radix[s++]) {
        const int R = plan.radix[s], m = L / (Ns * R);
        for (int r = 1; r < R; r++)
            for (int k = 0; k < Ns; k++) {
                const size_t a = 2 * (size_t(L) + Ns - 1 + size_t(r - 1) * Ns + k), b = 2 * size_t(r) * k * m;
                t[a] = t[b];
                t[a + 1] = t[b + 1];
            }
    }
    if (plan.chirp) {
        std::vector<T> ch(2 * size_t(N + L));
        std::vector<std::complex<long double>> b(L, 0.0L);
        for (long long k = 0; k < N; k++) {
            const auto c = root(k * k, 2LL * N);
            ch[2 * k] = T(c.real());
            ch[2 * k + 1] = T(c.imag());
            b[k] = b[(L - k) % L] = std::conj(c);
        }
        host_fft(b, roots);
        for (int k = 0; k < L; k++) {
            ch[2 * size_t(N + k)] = T(b[k].real() / L);
            ch[2 * size_t(N + k) + 1] = T(b[k].imag() / L);
        }
        if (hipMemcpy(chirp, ch.data(), ch.size() * sizeof(T), hipMemcpyHostToDevice) != hipSuccess)
            return VVM_ERR_HIP;
    }
    if (hipMemcpy(tw, t.data(), t.size() * sizeof(T), hipMemcpyHostToDevice) != hipSuccess) return VVM_ERR_HIP;
    hipLaunchKernelGGL(k_factor<T>, dim3(unsigned((Nq + 63) / 64)), dim3(64), 0, nullptr, N, M, cx, cu, di);
    cu_dev = cu;
    return hipStreamSynchronize(nullptr) == hipSuccess ? VVM_OK : VVM_ERR_HIP;
}

template <typename T>
void Direct<T>::destroy() {
    for (T *p : {tw, chirp, di, spec})
        if (p) (void)hipFree(p);
    tw = chirp = di = spec = nullptr;
}

template <typename T>
template <typename Mic>
void Direct<T>::columns(const Mic &mic, int nmic, hipStream_t st) {
    const dim3 gr(xcd_grid((plan.N + KC - 1) / KC).x + nmic);
    hipLaunchKernelGGL((k_columns<T, Mic>), gr, dim3(256), col_lds, st, plan.N, plan.M, spec, di, cu_dev, mic);
}

template <typename T>
template <bool C>
void Direct<T>::rows_solve(const double *r, const double *x0, double *x, const Grid &G, double *w, const double *rhow,
                           hipStream_t st) {
    const dim3 gr((plan.M + 1) / 2), b(plan.threads);
    hipLaunchKernelGGL((k_rows_fwd<T, false, C>), gr, b, row_lds, st, plan, tw, chirp, r, spec, Grid{}, StepPtrs{}, 0,
                       nullptr, Micro{});
    columns(NoMicro{}, 0, st);
    if (w)
        hipLaunchKernelGGL((k_rows_inv<T, true, true, C>), gr, b, row_lds, st, plan, tw, chirp, spec, x0, x, G, w,
                           rhow, nullptr);
    else if (x0)
        hipLaunchKernelGGL((k_rows_inv<T, true, false, C>), gr, b, row_lds, st, plan, tw, chirp, spec, x0, x, G,
                           nullptr, nullptr, nullptr);
    else
        hipLaunchKernelGGL((k_rows_inv<T, false, false, C>), gr, b, row_lds, st, plan, tw, chirp, spec, x0, x, G,
                           nullptr, nullptr, nullptr);
}
template <typename T>
void Direct<T>::solve(const double *r, const double *x0, double *x, hipStream_t st) {
    solve_w(r, x0, x, Grid{}, nullptr, nullptr, st);
}
template <typename T>
void Direct<T>::solve_w(const double *r, const double *x0, double *x, const Grid &G, double *w, const double *rhow,
                        hipStream_t st) {
    if (plan.chirp) rows_solve<true>(r, x0, x, G, w, rhow, st);
    else rows_solve<false>(r, x0, x, G, w, rhow, st);
}

template <typename T>
template <bool C>
void Direct<T>::rows_solve_step(const Grid &G, const StepPtrs &S, int step, const Micro *micro, double *f, double *x,
                                hipStream_t st) {
    const dim3 gr((plan.M + 1) / 2), b(plan.threads);
    Micro m;
    if (micro) {
        m = *micro;
        m.nblk = std::min(kMicroBlocks, micro_tiles(G, plan.threads));
    }
    hipLaunchKernelGGL((k_rows_fwd<T, true, C>), dim3(gr.x + (step >= 0 ? 1 : 0) + m.nblk), b, row_lds, st, plan, tw,
                       chirp, nullptr, spec, G, S, step, f, m);
    if (micro) {
        const int n = std::min(kMicroBlocks, micro_tiles(G, 256));
        columns(MicroPass{G, S, Negval{m.rs, m.nblk}, n}, n, st);
    } else {
        columns(NoMicro{}, 0, st);
    }
    hipLaunchKernelGGL((k_rows_inv<T, false, true, C>), gr, b, row_lds, st, plan, tw, chirp, spec, nullptr, x, G, S.w,
                       S.P.rhow, micro ? S.clock : nullptr);
}
template <typename T>
void Direct<T>::solve_step(const Grid &G, const StepPtrs &S, int step, const Micro *micro, double *f, double *x,
                           hipStream_t st) {
    if (plan.chirp) rows_solve_step<true>(G, S, step, micro, f, x, st);
    else rows_solve_step<false>(G, S, step, micro, f, x, st);
}

template class Direct<double>;
template class Direct<float>;

}  // namespace vvmd
