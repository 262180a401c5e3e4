// k_direct.hip -- direct solve of the cal_w system (direct.h).
//
// Three kernels: the forward row transforms, the tridiagonal systems, the
// inverse row transforms.  At 2048 x 255 they move 8 + 12 + 8 MB and are
// bound by latency (four LDS round trips a transform, the elimination's
// serial chain), not by bandwidth.
#include <algorithm>
#include <cmath>
#include <vector>

#include "direct.h"
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
template <int R, typename T>
__device__ inline void stage(T *re, T *im, int N, int Ns, const T *__restrict__ tw) {
    constexpr int NB = (8 + R - 1) / R;
    const int nb = N / R;
    Cx<T> v[NB][R];
    int dst[NB];
#pragma unroll
    for (int t = 0; t < NB; t++) {
        const int j = threadIdx.x + t * blockDim.x;
        if (j < nb) {
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
    }
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NB; t++) {
        if (int(threadIdx.x + t * blockDim.x) < nb) {
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

template <typename T>
__device__ inline void fft(const RowPlan &P, T *re, T *im, const T *__restrict__ tw, T *twl) {
    const int N = P.N;
    const T *tws = tw;
    if (P.tw_lds) {
        for (int t = threadIdx.x; t < 2 * N; t += blockDim.x) twl[t] = tw[t];
        tws = twl;
    }
    __syncthreads();
    int Ns = 1;
    for (int s = 0; s < P.nst; s++) {
        const int R = P.radix[s];
        // the stages' tables follow the table of all N roots; those before
        // hold sum (R - 1) Ns = Ns - 1 values
        const T *ts = tw + 2 * (N + Ns - 1);
        switch (R) {
            case 8: stage<8>(re, im, N, Ns, ts); break;
            case 4: stage<4>(re, im, N, Ns, ts); break;
            case 2: stage<2>(re, im, N, Ns, ts); break;
            case 3: stage<3>(re, im, N, Ns, ts); break;
            case 5: stage<5>(re, im, N, Ns, ts); break;
            default: stage_any(re, im, N, Ns, R, tws); break;
        }
        Ns *= R;
    }
}

// Hartley values (Re - Im) of the two rows at frequency q, from the complex
// spectrum Z of row a + i row b: A(q) = (Z(q) + Z*(N-q)) / 2,
// B(q) = (Z(q) - Z*(N-q)) / 2i.
template <typename T>
__device__ inline void hartley_pair(const T *re, const T *im, int N, int q, T &ha, T &hb) {
    const int a = pad(q), c = pad(q == 0 ? 0 : N - q);
    const T zr = re[a], zi = im[a], cr = re[c], ci = im[c];
    ha = T(0.5) * ((zr + cr) - (zi - ci));
    hb = T(0.5) * ((zi + ci) + (zr - cr));
}

// Forward: rows j, j+1 of r (RHS false), or cal_w's right-hand side
// f = -b / rhow, b = rhow^2 (zetap[i+1] - zetap[i]) dx
// (src/PoissonSolver.cpp:444-450), formed from zetap and stored (RHS true).
// With RHS and a step the last workgroup does pubarTop_pt instead: it reads u, w and K as
// the solve finds them, and alone it was a launch of 5 to 8 us.
template <typename T, bool RHS>
__global__ void __launch_bounds__(1024) k_rows_fwd(RowPlan P, const T *__restrict__ tw, const double *__restrict__ r,
                                                   T *__restrict__ spec, Grid G, StepPtrs S, int step,
                                                   double *__restrict__ f) {
    extern __shared__ unsigned char lds_raw[];
    if (RHS && step >= 0 && blockIdx.x == gridDim.x - 1) {
        pubartop_block(G, S, step);
        return;
    }
    const double *zetap = S.fut[F_ZETA], *rhow = S.P.rhow;
    const int N = P.N, M = P.M, LN = pad(N - 1) + 1;
    T *re = reinterpret_cast<T *>(lds_raw), *im = re + LN, *twl = im + LN;
    const int j = 1 + 2 * blockIdx.x;
    const bool two = j + 1 <= M;
    auto value = [&](int row, int i) -> double {
        if constexpr (!RHS) return r[size_t(row) * N + i];
        const int k = row + 1;
        const double rw = rhow[k];
        double v;
        {
#pragma clang fp contract(off)
            const double b = rw * rw * (zetap[ix(G, i + 2, k)] - zetap[ix(G, i + 1, k)]) * G.dx;
            v = -b / rw;
        }
        f[size_t(row) * N + i] = v;
        return v;
    };
#pragma unroll
    for (int t = 0; t < 8; t++) {  // threads >= N / 8; unrolled, all loads in flight at once
        const int i = threadIdx.x + t * blockDim.x;
        if (i < N) {
            re[pad(i)] = T(value(j, i));
            im[pad(i)] = two ? T(value(j + 1, i)) : T(0);
        }
    }
    fft(P, re, im, tw, twl);
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const int q = threadIdx.x + t * blockDim.x;
        if (q < N) {
            T ha, hb;
            hartley_pair(re, im, N, q, ha, hb);
            spec[size_t(j - 1) * N + q] = ha;
            if (two) spec[size_t(j) * N + q] = hb;
        }
    }
}

// Inverse: x = the transform of rows j, j+1 of spec (ADD: x0 + it); with w also
// w[i][k] = x / rhow[k] and BoundaryProcess2D_westdown(w)
// (src/PoissonSolver.cpp:469-476).
template <typename T, bool ADD, bool W>
__global__ void __launch_bounds__(1024) k_rows_inv(RowPlan P, const T *__restrict__ tw, const T *__restrict__ spec,
                                                   const double *x0, double *x, Grid G, double *__restrict__ w,
                                                   const double *__restrict__ rhow) {
    extern __shared__ unsigned char lds_raw[];
    const int N = P.N, M = P.M, LN = pad(N - 1) + 1;
    T *re = reinterpret_cast<T *>(lds_raw), *im = re + LN, *twl = im + LN;
    const int j = 1 + 2 * blockIdx.x;
    const bool two = j + 1 <= M;
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const int i = threadIdx.x + t * blockDim.x;
        if (i < N) {
            re[pad(i)] = spec[size_t(j - 1) * N + i];
            im[pad(i)] = two ? spec[size_t(j) * N + i] : T(0);
        }
    }
    if constexpr (W) {  // the zero rows of w
        for (int i = threadIdx.x; i < G.nx; i += blockDim.x) {
            if (blockIdx.x == 0) w[ix(G, i, 0)] = w[ix(G, i, 1)] = 0.;
            if (blockIdx.x == gridDim.x - 1) w[ix(G, i, G.nz - 1)] = 0.;
        }
    }
    fft(P, re, im, tw, twl);
    auto put = [&](int row, int i, T e) {
        const size_t a = size_t(row) * N + i;
        const double v = ADD ? x0[a] + double(e) : double(e);
        x[a] = v;
        if constexpr (W) store_westdown(w, G, i + 1, row + 1, v / rhow[row + 1]);
    };
#pragma unroll
    for (int t = 0; t < 8; t++) {
        const int q = threadIdx.x + t * blockDim.x;
        if (q < N) {
            T ha, hb;
            hartley_pair(re, im, N, q, ha, hb);
            put(j, q, ha);
            if (two) put(j + 1, q, hb);
        }
    }
}

// ------------------------------------------------------ tridiagonal systems
//
// Row j (1-based) of frequency q: d_j x_j - cu_j x_{j+1} - cu_{j-1} x_{j-1} =
// F_j.  Eliminated from both ends towards row mid = (M+1)/2 at once, which
// halves the serial chain:
//   downwards (j < mid): g_j = cu_j / p_j, y_{j+1} = F_{j+1} + g_j y_j,
//   upwards   (j > mid): g_j = cu_{j-1} / p_j, y_{j-1} = F_{j-1} + g_j y_j,
// x_mid = y_mid / p_mid, and back x_j = y_j / p_j + g_j x_{j+-1}.
// The factors g and 1 / (N p) (the inverse transform's 1/N folded in) are
// formed once, for q = 0..N/2 (lambda_q = lambda_{N-q}).

template <typename T>
__global__ void __launch_bounds__(64) k_factor(int N, int M, const double *__restrict__ cx,
                                               const double *__restrict__ cu, T *__restrict__ g, T *__restrict__ di) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x, Nq = N / 2 + 1;
    if (q >= Nq) return;
    const double s = sinpi(double(q) / N), lam = 4. * s * s;
    const int mid = (M + 1) / 2;
    auto diag = [&](int j) { return cx[j] * lam + cu[j] + cu[j - 1]; };
    double top = 0., bot = 0.;  // what the rows above and below take off p_mid
    for (int j = 1; j < mid; j++) {
        const double p = diag(j) - top, gj = cu[j] / p;
        g[size_t(j - 1) * Nq + q] = T(gj);
        di[size_t(j - 1) * Nq + q] = T(1. / (p * N));
        top = cu[j] * gj;
    }
    for (int j = M; j > mid; j--) {
        const double p = diag(j) - bot, gj = cu[j - 1] / p;
        g[size_t(j - 1) * Nq + q] = T(gj);
        di[size_t(j - 1) * Nq + q] = T(1. / (p * N));
        bot = cu[j - 1] * gj;
    }
    g[size_t(mid - 1) * Nq + q] = T(0);
    di[size_t(mid - 1) * Nq + q] = T(1. / ((diag(mid) - top - bot) * N));
}

// Eight columns a workgroup.  Every thread moves them and their factors to LDS
// in the order of the elimination's steps (all loads in flight at once): slot s
// of a direction holds its s-th row, after enough empty slots to make the
// number of steps a multiple of eight.  Then 16 lanes, 8 columns x 2
// directions, run all steps without a branch, the next eight steps' values in
// registers; an empty slot leaves y = 0 and x is not read after it.
// At 2048 x 255: 15 us; with the rows in place and the two directions'
// last steps under a mask 27 us.
constexpr int KC = 8, KSTEP = 8, KL = 2 * KC;
struct ColSteps {
    int mid, steps, pad_dn, pad_up;
};
__host__ __device__ inline ColSteps col_steps(int M) {
    ColSteps c;
    c.mid = (M + 1) / 2 - 1;  // 0-based
    const int dn = c.mid, up = M - 1 - c.mid;
    c.steps = ((dn > up ? dn : up) + KSTEP - 1) / KSTEP * KSTEP;
    c.pad_dn = c.steps - dn;
    c.pad_up = c.steps - up;
    return c;
}
// LDS elements: [steps][F, g, 1/p][KL], then the middle row's F and 1/p
inline size_t col_lds_elems(int M) { return size_t(col_steps(M).steps) * 3 * KL + 2 * KC; }

template <typename T>
__global__ void __launch_bounds__(256) k_columns(int N, int M, T *__restrict__ spec, const T *__restrict__ g,
                                                 const T *__restrict__ di) {
    extern __shared__ unsigned char lds_raw[];
    T *L = reinterpret_cast<T *>(lds_raw);
    const ColSteps cs = col_steps(M);
    T *Mid = L + size_t(cs.steps) * 3 * KL;
    const int Nq = N / 2 + 1;
    // columns past the last repeat it (never stored)
    const int c = threadIdx.x % KC, q = min(int(blockIdx.x) * KC + c, N - 1), qq = min(q, N - q);
    const int rstep = blockDim.x / KC;
    // element of row j (0-based, not mid) in L
    auto slot = [&](int j) {
        return j < cs.mid ? (cs.pad_dn + j) * 3 * KL + c : (cs.pad_up + M - 1 - j) * 3 * KL + KC + c;
    };
    for (int j0 = threadIdx.x / KC; j0 < M; j0 += 8 * rstep) {
        T vf[8], vg[8], vd[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int j = min(j0 + u * rstep, M - 1);
            vf[u] = spec[size_t(j) * N + q];
            vg[u] = g[size_t(j) * Nq + qq];
            vd[u] = di[size_t(j) * Nq + qq];
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int j = j0 + u * rstep;
            if (j < M && j != cs.mid) {
                T *p = L + slot(j);
                p[0] = vf[u];
                p[KL] = vg[u];
                p[2 * KL] = vd[u];
            } else if (j == cs.mid) {
                Mid[c] = vf[u];
                Mid[KC + c] = vd[u];
            }
        }
    }
    for (int t = threadIdx.x; t < cs.pad_dn * 3 * KL; t += blockDim.x)
        if (t % KL < KC) L[t] = T(0);
    for (int t = threadIdx.x; t < cs.pad_up * 3 * KL; t += blockDim.x)
        if (t % KL >= KC) L[t] = T(0);
    __syncthreads();
    if (threadIdx.x < KL) {
        T *p = L + threadIdx.x;
        T y = T(0), gp = T(0);
        T nf[KSTEP], ng[KSTEP], nd[KSTEP];
#pragma unroll
        for (int u = 0; u < KSTEP; u++) {
            nf[u] = p[u * 3 * KL];
            ng[u] = p[u * 3 * KL + KL];
            nd[u] = p[u * 3 * KL + 2 * KL];
        }
        for (int s = 0; s < cs.steps; s += KSTEP, p += KSTEP * 3 * KL) {
            T vf[KSTEP], vg[KSTEP], vd[KSTEP];
#pragma unroll
            for (int u = 0; u < KSTEP; u++) {
                vf[u] = nf[u];
                vg[u] = ng[u];
                vd[u] = nd[u];
            }
            // past the last step this reads the same eight again
            const T *nx = s + KSTEP < cs.steps ? p + KSTEP * 3 * KL : p;
#pragma unroll
            for (int u = 0; u < KSTEP; u++) {
                nf[u] = nx[u * 3 * KL];
                ng[u] = nx[u * 3 * KL + KL];
                nd[u] = nx[u * 3 * KL + 2 * KL];
            }
#pragma unroll
            for (int u = 0; u < KSTEP; u++) {
                y = vf[u] + gp * y;
                gp = vg[u];
                vf[u] = y * vd[u];
            }
#pragma unroll
            for (int u = 0; u < KSTEP; u++) p[u * 3 * KL] = vf[u];
        }
        const int col = threadIdx.x % KC;
        const bool up = threadIdx.x >= KC;
        const T off = gp * y, other = __shfl_xor(off, KC, kWave);
        // the same order of terms in both directions' lanes
        T x = (Mid[col] + (up ? other : off) + (up ? off : other)) * Mid[KC + col];
        if (!up) Mid[col] = x;
        p -= KSTEP * 3 * KL;
#pragma unroll
        for (int u = 0; u < KSTEP; u++) {
            nf[u] = p[u * 3 * KL];
            ng[u] = p[u * 3 * KL + KL];
        }
        for (int s = cs.steps; s > 0; s -= KSTEP, p -= KSTEP * 3 * KL) {
            T vf[KSTEP], vg[KSTEP];
#pragma unroll
            for (int u = 0; u < KSTEP; u++) {
                vf[u] = nf[u];
                vg[u] = ng[u];
            }
            const T *nx = s > KSTEP ? p - KSTEP * 3 * KL : p;
#pragma unroll
            for (int u = 0; u < KSTEP; u++) {
                nf[u] = nx[u * 3 * KL];
                ng[u] = nx[u * 3 * KL + KL];
            }
#pragma unroll
            for (int u = KSTEP - 1; u >= 0; u--) {
                x = vf[u] + vg[u] * x;
                vf[u] = x;
            }
#pragma unroll
            for (int u = 0; u < KSTEP; u++) p[u * 3 * KL] = vf[u];
        }
    }
    __syncthreads();
    if (int(blockIdx.x) * KC + c >= N) return;
    for (int j = threadIdx.x / KC; j < M; j += rstep) spec[size_t(j) * N + q] = j == cs.mid ? Mid[c] : L[slot(j)];
}

constexpr size_t kLdsMax = 160 * 1024;

template <typename T>
T *dalloc(size_t n) {
    void *p = nullptr;
    if (hipMalloc(&p, n * sizeof(T)) != hipSuccess) return nullptr;
    return static_cast<T *>(p);
}

template <typename K>
bool allow_lds(K kernel, size_t bytes) {
    return bytes <= 64 * 1024 || hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize,
                                                     int(bytes)) == hipSuccess;
}

}  // namespace

template <typename T>
int Direct<T>::init(int N, int M, const double *cx, const double *cu) {
    plan = RowPlan();
    plan.N = N;
    plan.M = M;
    int n = N;
    for (int r : {8, 4, 2, 3, 5})
        while (n % r == 0 && plan.nst < kMaxStages) {
            plan.radix[plan.nst++] = r;
            n /= r;
        }
    bool other = false;
    for (int r = 7; n > 1 && plan.nst < kMaxStages; r += 2) {
        if (r * r > n) r = n;
        while (n % r == 0 && plan.nst < kMaxStages) {
            plan.radix[plan.nst++] = r;
            n /= r;
            other = true;
        }
    }
    if (n != 1 || N > 8192) return VVM_ERR_SIZE;
    plan.threads = std::min(1024, std::max(64, ((N + 7) / 8 + 63) / 64 * 64));
    const size_t LN = size_t(N - 1) + size_t((N - 1) >> 5) + 1;
    row_lds = 2 * LN * sizeof(T);
    if (other && row_lds + 2 * size_t(N) * sizeof(T) <= kLdsMax) {
        plan.tw_lds = 1;
        row_lds += 2 * size_t(N) * sizeof(T);
    }
    col_lds = col_lds_elems(M) * sizeof(T);
    if (row_lds > kLdsMax || col_lds > kLdsMax) return VVM_ERR_SIZE;
    if (!allow_lds(k_rows_fwd<T, false>, row_lds) || !allow_lds(k_rows_fwd<T, true>, row_lds) ||
        !allow_lds(k_rows_inv<T, false, false>, row_lds) || !allow_lds(k_rows_inv<T, true, false>, row_lds) ||
        !allow_lds(k_rows_inv<T, false, true>, row_lds) || !allow_lds(k_columns<T>, col_lds))
        return VVM_ERR_HIP;
    const size_t Nq = size_t(N) / 2 + 1;
    tw = dalloc<T>(4 * size_t(N));
    g = dalloc<T>(Nq * M);
    di = dalloc<T>(Nq * M);
    spec = dalloc<T>(size_t(N) * M);
    if (!tw || !g || !di || !spec) {
        destroy();
        return VVM_ERR_NOMEM;
    }
    std::vector<T> t(4 * size_t(N), T(0));
    for (int k = 0; k < N; k++) {
        const long double a = 2.0L * 3.14159265358979323846264338327950288L * k / N;
        t[2 * k] = T(std::cos(a));
        t[2 * k + 1] = T(-std::sin(a));
    }
    // the stages' twiddles, picked from those (r k < Ns R, so r k N / (Ns R) < N)
    for (int s = 0, Ns = 1; s < plan.nst; Ns *= plan.radix[s++]) {
        const int R = plan.radix[s], m = N / (Ns * R);
        for (int r = 1; r < R; r++)
            for (int k = 0; k < Ns; k++) {
                const size_t a = 2 * (size_t(N) + Ns - 1 + size_t(r - 1) * Ns + k), b = 2 * size_t(r) * k * m;
                t[a] = t[b];
                t[a + 1] = t[b + 1];
            }
    }
    if (hipMemcpy(tw, t.data(), t.size() * sizeof(T), hipMemcpyHostToDevice) != hipSuccess) return VVM_ERR_HIP;
    hipLaunchKernelGGL(k_factor<T>, dim3(unsigned((Nq + 63) / 64)), dim3(64), 0, nullptr, N, M, cx, cu, g, di);
    return hipStreamSynchronize(nullptr) == hipSuccess ? VVM_OK : VVM_ERR_HIP;
}

template <typename T>
void Direct<T>::destroy() {
    for (T *p : {tw, g, di, spec})
        if (p) (void)hipFree(p);
    tw = g = di = spec = nullptr;
}

template <typename T>
void Direct<T>::columns(hipStream_t st) {
    hipLaunchKernelGGL(k_columns<T>, dim3((plan.N + KC - 1) / KC), dim3(256), col_lds, st, plan.N, plan.M, spec, g,
                       di);
}

template <typename T>
void Direct<T>::solve(const double *r, const double *x0, double *x, hipStream_t st) {
    const dim3 gr((plan.M + 1) / 2), b(plan.threads);
    hipLaunchKernelGGL((k_rows_fwd<T, false>), gr, b, row_lds, st, plan, tw, r, spec, Grid{}, StepPtrs{}, 0,
                       nullptr);
    columns(st);
    if (x0)
        hipLaunchKernelGGL((k_rows_inv<T, true, false>), gr, b, row_lds, st, plan, tw, spec, x0, x, Grid{}, nullptr,
                           nullptr);
    else
        hipLaunchKernelGGL((k_rows_inv<T, false, false>), gr, b, row_lds, st, plan, tw, spec, x0, x, Grid{}, nullptr,
                           nullptr);
}

template <typename T>
void Direct<T>::solve_step(const Grid &G, const StepPtrs &S, int step, double *f, double *x, hipStream_t st) {
    const dim3 gr((plan.M + 1) / 2), b(plan.threads);
    hipLaunchKernelGGL((k_rows_fwd<T, true>), dim3(gr.x + (step >= 0 ? 1 : 0)), b, row_lds, st, plan, tw, nullptr, spec, G, S, step, f);
    columns(st);
    hipLaunchKernelGGL((k_rows_inv<T, false, true>), gr, b, row_lds, st, plan, tw, spec, nullptr, x, G, S.w,
                       S.P.rhow);
}

template class Direct<double>;
template class Direct<float>;

}  // namespace vvmd
