// k_poisson.hip -- the elliptic part of a VVM timestep on the device:
// PoissonSolver::cal_w (src/PoissonSolver.cpp:439-477) by the direct solver
// (k_direct.hip) with FP64 iterative refinement, or as multigrid-
// preconditioned CG in FP64, and PoissonSolver::cal_u
// (src/PoissonSolver.cpp:580-653).
//
// Multigrid: geometric, vertex coarsening (N -> N/2 periodic columns,
// M -> (M-1)/2 Dirichlet rows), operators rediscretised with harmonic-mean
// vertical conductances, bilinear prolongation P and restriction P^T,
// damped-Jacobi V(2,2) smoothing and a single-workgroup coarsest solve.
// Every piece is symmetric, so the V-cycle is a valid CG preconditioner.
#pragma clang fp contract(off)

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "poisson.h"

namespace vvmd {

namespace {

constexpr int LX = 64, LY = 4;

inline dim3 lgrid(int N, int M) { return dim3((N + LX - 1) / LX, (M + LY - 1) / LY); }

template <typename T>
__device__ inline T applyL(const T *__restrict__ x, int N, int i, int j, T cxj, T cuj, T cujm) {
    const int im = (i == 0) ? N - 1 : i - 1, ip = (i == N - 1) ? 0 : i + 1;
    const size_t r = size_t(j) * N;
    const T c = x[r + i];
    return cxj * (T(2) * c - x[r + im] - x[r + ip]) + cuj * (c - x[r + N + i]) + cujm * (c - x[r - N + i]);
}

// ------------------------------------------------------------------ CG

// The two CG vector kernels run on at most kCGBlocks workgroups, each
// walking LX x LY tiles, so that the update kernel can add the p.q partials
// of every pq workgroup itself (no k_finalize between them).
constexpr int kCGBlocks = 1024;
inline int cg_blocks(int N, int M) { return std::min(kCGBlocks, int(nblocks(lgrid(N, M)))); }

// p = z + beta p (beta = 0 on the first iteration), q = L p, partials of p.q
// into rs_pq.  After the first iteration every workgroup adds the n_rz
// partials of r.z the preconditioner left in rs_rz, beta = r.z / sc[old];
// workgroup 0 stores r.z in sc[fresh] for the update.
template <typename T>
__global__ void __launch_bounds__(LX *LY) k_pcg_pq(int N, int M, const T *z, const T *pin, T *pout, T *q, const T *cx,
                                                   const T *cu, double *sc, RedSlot rs_pq, int first, RedSlot rs_rz,
                                                   int n_rz, int old, int fresh) {
    const int tiles_x = (N + LX - 1) / LX, ntiles = tiles_x * ((M + LY - 1) / LY);
    T beta = T(0);
    if (!first) {
        const double rz = block_total(rs_rz, n_rz);
        beta = T(rz / sc[old]);
        if (blockIdx.x == 0 && threadIdx.x == 0 && threadIdx.y == 0) sc[fresh] = rz;
    }
    double part[1] = {0.};
    for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const int i = (t % tiles_x) * LX + threadIdx.x, j = 1 + (t / tiles_x) * LY + threadIdx.y;
        if (i < N && j <= M) {
            const int im = (i == 0) ? N - 1 : i - 1, ip = (i == N - 1) ? 0 : i + 1;
            const size_t r = size_t(j) * N;
            auto pn = [&](size_t a) -> T { return first ? z[a] : z[a] + beta * pin[a]; };
            const T c = pn(r + i);
            const T Lp = cx[j] * (T(2) * c - pn(r + im) - pn(r + ip)) + cu[j] * (c - pn(r + N + i)) +
                         cu[j - 1] * (c - pn(r - N + i));
            pout[r + i] = c;
            q[r + i] = Lp;
            part[0] += double(c) * double(Lp);
        }
    }
    block_partials<1>(part, rs_pq);
}

// alpha = sc[rz] / p.q (p.q from the npq partials of k_pcg_pq), x += alpha p,
// r -= alpha q, and ||w r||^2 with the row weights w (rhow: the reference
// system's residual) as partials in rs.
template <typename T>
__global__ void __launch_bounds__(LX *LY) k_pcg_update(int N, int M, T *x, T *r, const T *p, const T *q,
                                                       const T *wD, double *sc, int rz, RedSlot rs_pq, int npq,
                                                       RedSlot rs) {
    const int tiles_x = (N + LX - 1) / LX, ntiles = tiles_x * ((M + LY - 1) / LY);
    const T alpha = T(sc[rz] / block_total(rs_pq, npq));
    double part[1] = {0.};
    for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
        const int i = (t % tiles_x) * LX + threadIdx.x, j = 1 + (t / tiles_x) * LY + threadIdx.y;
        if (i < N && j <= M) {
            const size_t c = size_t(j) * N + i;
            x[c] = x[c] + alpha * p[c];
            const T rn = r[c] - alpha * q[c];
            r[c] = rn;
            const double wr = double(wD[j]) * double(rn);
            part[0] += wr * wr;
        }
    }
    block_partials<1>(part, rs);
}

// The solve's first residual with the guess folded in.  XF_EXTRAP: x = the
// extrapolation of order ord (2 x1 - x2, or 3 (x1 - x2) + x3), XF_ZERO:
// x = 0, XF_NONE: x as it is.  Every value of x the stencil needs is formed
// on the fly with the same arithmetic the separate kernels used, so r and x
// are bit for bit what they gave.
enum { XF_NONE = 0, XF_EXTRAP, XF_ZERO };
template <int XF>
__global__ void __launch_bounds__(LX *LY) k_residual_x(int N, int M, const double *f, double *x, const double *x1,
                                                       const double *x2, const double *x3, int ord, double *r,
                                                       const double *cx, const double *cu, const double *wD,
                                                       RedSlot rs) {
    const int i = blockIdx.x * LX + threadIdx.x, j = 1 + blockIdx.y * LY + threadIdx.y;
    auto xv = [&](size_t a) -> double {
        if (XF == XF_EXTRAP) return extrap_at(x1, x2, x3, ord, a);
        if (XF == XF_ZERO) return 0.;
        return x[a];
    };
    double part[1] = {0.};
    if (i < N && j <= M) {
        const size_t c = size_t(j) * N + i;
        const int im = (i == 0) ? N - 1 : i - 1, ip = (i == N - 1) ? 0 : i + 1;
        const size_t rw = size_t(j) * N;
        const double xc = xv(rw + i);
        const double Lx = cx[j] * (2. * xc - xv(rw + im) - xv(rw + ip)) + cu[j] * (xc - xv(rw + N + i)) +
                          cu[j - 1] * (xc - xv(rw - N + i));
        const double rv = f[c] - Lx;
        r[c] = rv;
        if (XF != XF_NONE) {
            x[c] = xc;
            if (j == 1) x[i] = xv(i);
            if (j == M) x[rw + N + i] = xv(rw + N + i);
        }
        const double wr = wD[j] * rv;
        part[0] = wr * wr;
    }
    block_partials<1>(part, rs);
}

// ------------------------------------------------------------- cal_w glue

// b = rhow^2 (zetap[i+1] - zetap[i]) dx (src/PoissonSolver.cpp:444-450) for
// k = 2..nz-2 and f = -b / rhow; ||b||^2 into sc[P_BNORM2].
__global__ void __launch_bounds__(LX *LY) k_calw_rhs(Grid G, const double *zetap, const double *rhow, double *f,
                                                     double *sc, RedSlot rs) {
    const int N = G.nx - 2, M = G.nz - 3;
    const int ii = blockIdx.x * LX + threadIdx.x, j = 1 + blockIdx.y * LY + threadIdx.y;
    double part[1] = {0.};
    if (ii < N && j <= M) {
        const int i = ii + 1, k = j + 1;
        const double b = rhow[k] * rhow[k] * (zetap[ix(G, i + 1, k)] - zetap[ix(G, i, k)]) * G.dx;
        f[size_t(j) * N + ii] = -b / rhow[k];
        part[0] = b * b;
    }
    block_partials<1>(part, rs);
}

__global__ void __launch_bounds__(LX *LY) k_rhs_from_b(int N, int M, const double *bref, const double *wD,
                                                       double *f, double *sc, RedSlot rs) {
    const int ii = blockIdx.x * LX + threadIdx.x, j = 1 + blockIdx.y * LY + threadIdx.y;
    double part[1] = {0.};
    if (ii < N && j <= M) {
        const double b = bref[size_t(j - 1) * N + ii];
        f[size_t(j) * N + ii] = -b / wD[j];
        part[0] = b * b;
    }
    block_partials<1>(part, rs);
}

__global__ void k_x_ref(int N, int M, double *x, double *xref, int to_ref) {
    const int ii = blockIdx.x * LX + threadIdx.x, j = 1 + blockIdx.y * LY + threadIdx.y;
    if (ii >= N || j > M) return;
    if (to_ref) xref[size_t(j - 1) * N + ii] = x[size_t(j) * N + ii];
    else x[size_t(j) * N + ii] = xref[size_t(j - 1) * N + ii];
}

// w[i][k] = x / rhow[k] and BoundaryProcess2D_westdown(w) (:469-476).
__global__ void __launch_bounds__(LX *LY) k_calw_back(Grid G, const double *x, double *w, const double *rhow) {
    const int i = blockIdx.x * LX + threadIdx.x, k = blockIdx.y * LY + threadIdx.y;
    if (i >= G.nx || k >= G.nz) return;
    if (k == 0 || k == 1 || k == G.nz - 1) {
        w[ix(G, i, k)] = 0.;
        return;
    }
    if (i < 1 || i > G.nx - 2) return;
    const int N = G.nx - 2;
    store_westdown(w, G, i, k, x[size_t(k - 1) * N + (i - 1)] / rhow[k]);
}

__global__ void k_extrapolate(size_t n, double *x, const double *x1, const double *x2, const double *x3, int ord) {
    const size_t t = size_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (t >= n) return;
    x[t] = extrap_at(x1, x2, x3, ord, t);
}

// ------------------------------------------------------------------ cal_u

// Over 1024 threads (16 wavefronts): the exclusive prefix sum of v, its total
// and that of t.
__device__ inline double block_excl_sum(double v, double t, double *total, double *ttotal) {
    __shared__ double ws[2][16];
    const int lane = threadIdx.x % kWave, wid = uniform(threadIdx.x / kWave);
    const double inc = wave_scan(v), below = dpp<DPP_WAVE_SHR1>(inc), tw = wave_scan(t);
    if (lane == kWave - 1) {
        ws[0][wid] = inc;
        ws[1][wid] = tw;
    }
    __syncthreads();
    const double s = row_scan(ws[lane / 16 % 2][lane % 16]);
    __syncthreads();
    *total = from_lane(s, 15);
    *ttotal = from_lane(s, 31);
    return wid > 0 ? from_lane(s, wid - 1) + below : below;
}

// The residual's norms, one pair of partial sums per workgroup: block of nblk
// 1024-thread workgroups, each walking 64 x 16 tiles, four tiles' loads in
// flight (a thread outside the grid reads its edge).
__device__ inline void residual_norms(const Residual &R, int block, int nblk) {
    constexpr int RX = 64, RY = 16, U = 4;
    const int N = R.N, M = R.M, tx = (N + RX - 1) / RX, nt = tx * ((M + RY - 1) / RY);
    double part[2] = {0., 0.};
    for (int t0 = block; t0 < nt; t0 += U * nblk) {
        double fv[U], lv[U], wd[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (u > 0 && t0 + u * nblk >= nt) break;
            const int t = t0 + u * nblk;
            const int i = min((t % tx) * RX + int(threadIdx.x % RX), N - 1);
            const int j = min(1 + (t / tx) * RY + uniform(threadIdx.x / RX), M);
            fv[u] = R.f[size_t(j) * N + i];
            lv[u] = applyL(R.x, N, i, j, R.cx[j], R.cu[j], R.cu[j - 1]);
            wd[u] = R.wD[j];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int t = t0 + u * nblk;
            const int i = (t % tx) * RX + threadIdx.x % RX, j = 1 + (t / tx) * RY + threadIdx.x / RX;
            if (t < nt && i < N && j <= M) {
                const double wr = wd[u] * (fv[u] - lv[u]), wb = wd[u] * fv[u];
                part[0] += wr * wr;
                part[1] += wb * wb;
            }
        }
    }
    block_sum<2>(part);
    if (threadIdx.x == 0) {
        __hip_atomic_store(R.hres + 2 * block, part[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(R.hres + 2 * block + 1, part[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// r = f - L x and the norms, before a correction.  FIRST: the right-hand side
// and the guess in the reference's order (bref, xref), f and x formed on the
// way: four passes in one.
template <bool FIRST>
__global__ void __launch_bounds__(1024) k_solve_residual(Residual R, const double *__restrict__ bref,
                                                         const double *__restrict__ xref, double *__restrict__ f,
                                                         double *__restrict__ x, double *__restrict__ r) {
    constexpr int RX = 64, RY = 16;
    const int N = R.N, M = R.M, tx = (N + RX - 1) / RX, nt = tx * ((M + RY - 1) / RY);
    double part[2] = {0., 0.};
#pragma unroll 2
    for (int t = blockIdx.x; t < nt; t += gridDim.x) {
        const int i = (t % tx) * RX + threadIdx.x % RX, j = 1 + (t / tx) * RY + uniform(threadIdx.x / RX);
        if (j > M) continue;
        const int ic = min(i, N - 1), im = ic == 0 ? N - 1 : ic - 1, ip = ic == N - 1 ? 0 : ic + 1;
        const size_t c = size_t(j) * N + ic;
        double xc, xw, xe, xu, xd, fv, wb;
        if constexpr (FIRST) {
            const double *row = xref + size_t(j - 1) * N;  // rows 0 and M + 1 are zero
            xc = row[ic], xw = row[im], xe = row[ip];
            xu = j < M ? row[N + ic] : 0.;
            xd = j > 1 ? row[ic - N] : 0.;
            wb = bref[size_t(j - 1) * N + ic];
            fv = -wb / R.wD[j];
        } else {
            const double *row = R.x + size_t(j) * N;
            xc = row[ic], xw = row[im], xe = row[ip], xu = row[N + ic], xd = row[ic - N];
            fv = R.f[c];
            wb = R.wD[j] * fv;
        }
        const double rv = fv - (R.cx[j] * (2. * xc - xw - xe) + R.cu[j] * (xc - xu) + R.cu[j - 1] * (xc - xd));
        const double wr = R.wD[j] * rv;
        if (i < N) {
            r[c] = rv;
            if constexpr (FIRST) {
                f[c] = fv;
                x[c] = xc;
            }
            part[0] += wr * wr;
            part[1] += wb * wb;
        }
    }
    block_sum<2>(part);
    if (threadIdx.x == 0) {
        __hip_atomic_store(R.hres + 2 * blockIdx.x, part[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        __hip_atomic_store(R.hres + 2 * blockIdx.x + 1, part[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// cal_u.  Top row: h (mean removed), the periodic 1-D problem G y = h solved
// in closed form through its first differences D_r = y_r - y_{r-1}:
// D_{r+1} - D_r = h_r and sum_r D_r = 0, so D_r = S_r - mean(S) with S the
// exclusive prefix sum of h.  uxi = D rdx (mean removed as in the
// reference), u[i][nz-2] = uxi + ubarTopp, and xi = the mean-free y.  With P
// the prefix sum of h as it is, S_r = P_r - r mean(h), and sum_r S_r =
// sum_r ((N-1)/2 - r) h_r, which the scan of h brings along.
//
// Then the downward integration u[i][k] = u[i][nz-2] - dz sum_{k'=k}^{nz-3}
// ((w[i][k'+1]-w[i-1][k'+1]) rdx - rhow[k'+1] zetap[i][k'+1]) (:643-650):
// UW columns x UC vertical chunks per block (narrow blocks, so that there are
// enough workgroups for every CU), chunk sums scanned in LDS.
//
// Every workgroup forms the whole top row's prefix sums for its own 16
// columns, two block scans that take 1.6 us at 1024 columns (three, through LDS
// shuffles, 4.5): cheaper than a kernel of one workgroup before this one (13
// us at 2048 columns, 11 at 128).  The rest is the latency of the first loads,
// 3 us there; a chunk's levels, up to UT, are read once and kept.  64 registers
// at most, so that a CU holds two workgroups and 4096 columns run in one round.
// The workgroups from ncol on form the residual norms of the solve that left
// w, which would be a launch of 4 to 5 us.
constexpr int UW = 16, UC = 64, UT = 4;
__global__ void __launch_bounds__(UW *UC) __attribute__((amdgpu_waves_per_eu(8))) k_calu(Grid G, StepPtrs S, int ncol, Residual R) {
    extern __shared__ double sh[];  // N doubles: P
    __shared__ double cs[UW * UC / kWave][UW], top[UW];
    if (int(blockIdx.x) >= ncol) {
        residual_norms(R, blockIdx.x - ncol, gridDim.x - ncol);
        note_end(S.clock, CLK_SOLVE_END);
        return;
    }
    const int N = G.nx - 2, nz = G.nz, tid = threadIdx.x;
    const double *w = S.w, *zp = S.fut[F_ZETA], *rhow = S.P.rhow, *rhou = S.P.rhou;
    const int i = 1 + blockIdx.x * UW + tid % UW, c = tid / UW, ic = min(i, N);
    const int K = nz - 3;  // levels nz-3 .. 1
    const int C = (K + UC - 1) / UC;
    const bool col = (i <= N);
    const int E = (N + UW * UC - 1) / (UW * UC), r0 = min(tid * E, N), r1 = min(r0 + E, N);
    // every load before the first wait: the top row, and up to UT levels of
    // the thread's chunk
    double hv[8], tv[UT];
#pragma unroll
    for (int e = 0; e < 8; e++)  // N <= 8 UW UC
        if (e < E) hv[e] = w[ix(G, 1 + min(tid + e * UW * UC, N - 1), nz - 2)];
    auto term = [&](int k) {  // level k's part of the integral
        return ((w[ix(G, ic, k + 1)] - w[ix(G, ic - 1, k + 1)]) * G.rdx - rhow[k + 1] * zp[ix(G, ic, k + 1)]) * -G.dz;
    };
    const int kk0 = min(c * C, K), kk1 = min(kk0 + C, K);
#pragma unroll
    for (int u = 0; u < UT; u++)
        if (u < C) tv[u] = term(max(nz - 3 - (kk0 + u), 1));
    const double ubp = S.s[S_UBARTOPP];
#pragma unroll
    for (int e = 0; e < 8; e++)
        if (e < E && tid + e * UW * UC < N)  // src/PoissonSolver.cpp:585-594
            sh[tid + e * UW * UC] = -(0. - rhow[nz - 2] * hv[e]) / rhou[nz - 2] * G.dx;
    // the chunk's sum; the sums of the wavefront's chunks above it (four, 16
    // lanes apart), and the wavefront's to LDS
    double loc = 0.;
#pragma unroll
    for (int u = 0; u < UT; u++)
        if (kk0 + u < kk1) loc += tv[u];
    for (int kk = kk0 + UT; kk < kk1; kk++) loc += term(nz - 3 - kk);
    double above = 0.;
#pragma unroll
    for (int d = 1; d < kWave / UW; d++) {
        const double o = __shfl_up(loc, d * UW, kWave);
        if (tid % kWave >= d * UW) above += o;
    }
    if (tid % kWave >= kWave - UW) cs[tid / kWave][tid % UW] = above + loc;
    __syncthreads();

    loc = 0.;
    double mom = 0.;  // sum over r of S_r
    for (int r = r0; r < r1; r++) {
        loc += sh[r];
        mom += (0.5 * (N - 1) - r) * sh[r];
    }
    double tot, sm;
    double p = block_excl_sum(loc, mom, &tot, &sm);
    const double hm = tot / N;
    sm /= N;
    for (int r = r0; r < r1; r++) {
        const double h = sh[r];
        sh[r] = p;
        p += h;
    }
    auto D = [&](int r) { return sh[r] - r * hm - sm; };
    double sd = 0., none;
    for (int r = r0; r < r1; r++) sd += D(r);
    double y = block_excl_sum(sd, 0., &tot, &none);
    const double um = tot * G.rdx / N;  // :621-634
    const int b0 = blockIdx.x * UW;
    for (int r = max(r0, b0); r < min(r1, b0 + UW); r++) {
        const double uxi = D(r) * G.rdx - um;
        S.uxi[r + 1] = uxi;
        if (r + 1 == N) S.uxi[0] = uxi;
        if (r == 0) S.uxi[N + 1] = uxi;
        top[r - b0] = uxi + ubp;
        store_center(S.u, G, r + 1, nz - 2, uxi + ubp);
    }
    if (blockIdx.x == 0) {
        // xi: y_r = sum_{j<=r} D_j minus its mean (min-norm solution); what
        // rounding left of D's own mean would grow with r
        const double dm = tot / N;
        y -= r0 * dm;
        double sy = 0., yr = y;
        for (int r = r0; r < r1; r++) {
            yr += D(r) - dm;
            sy += yr;
        }
        block_excl_sum(sy, 0., &tot, &none);
        const double ym = tot / N;
        yr = y;
        for (int r = r0; r < r1; r++) {
            yr += D(r) - dm;
            const double xi = yr - ym;
            S.xi[r + 1] = xi;
            if (r + 1 == N) S.xi[0] = xi;
            if (r == 0) S.xi[N + 1] = xi;
        }
    }
    __syncthreads();  // top
    if (!col) return;
    double area = 0.;
    for (int w2 = 0; w2 < tid / kWave; w2++) area += cs[w2][tid % UW];
    area += above;
    const double utop = top[tid % UW];
#pragma unroll
    for (int u = 0; u < UT; u++)
        if (kk0 + u < kk1) {
            area += tv[u];
            store_center(S.u, G, i, nz - 3 - (kk0 + u), area + utop);
        }
    for (int kk = kk0 + UT; kk < kk1; kk++) {
        area += term(nz - 3 - kk);
        store_center(S.u, G, i, nz - 3 - kk, area + utop);
    }
}

template <typename T>
T *dalloc(size_t n) {
    void *p = nullptr;
    if (hipMalloc(&p, n * sizeof(T)) != hipSuccess) return nullptr;
    hipMemset(p, 0, n * sizeof(T));
    return static_cast<T *>(p);
}

template <typename T>
bool build_hier(MGHier<T> &H, int N, int M, const std::vector<double> &cx0, const std::vector<double> &cu0) {
    std::vector<double> cx = cx0, cu = cu0;
    int l = 0;
    while (true) {
        MGLevel<T> &L = H.lev[l];
        L.N = N;
        L.M = M;
        std::vector<T> tcx(M + 2, T(0)), tcu(M + 1), tdi(M + 2, T(0));
        for (int j = 0; j <= M + 1; j++) tcx[j] = T(cx[j]);
        for (int j = 0; j <= M; j++) tcu[j] = T(cu[j]);
        for (int j = 1; j <= M; j++) tdi[j] = T(1. / (2. * cx[j] + cu[j] + cu[j - 1]));
        L.cx = dalloc<T>(M + 2);
        L.cu = dalloc<T>(M + 1);
        L.dinv = dalloc<T>(M + 2);
        if (!L.cx || !L.cu || !L.dinv) return false;
        hipMemcpy(L.cx, tcx.data(), sizeof(T) * (M + 2), hipMemcpyHostToDevice);
        hipMemcpy(L.cu, tcu.data(), sizeof(T) * (M + 1), hipMemcpyHostToDevice);
        hipMemcpy(L.dinv, tdi.data(), sizeof(T) * (M + 2), hipMemcpyHostToDevice);
        if (l > 0) {
            const size_t n = size_t(M + 2) * N;
            L.x = dalloc<T>(n);
            L.b = dalloc<T>(n);
            L.t = dalloc<T>(n);
            if (!L.x || !L.b || !L.t) return false;
        }
        l++;
        const bool can = (M >= 3) && (M % 2 == 1) && (N >= 4) && (N % 2 == 0) && (l < kMaxLevels);
        if (!can) break;
        const int Mc = (M - 1) / 2, Nc = N / 2;
        std::vector<double> ccx(Mc + 2, 0.), ccu(Mc + 1);
        for (int jc = 1; jc <= Mc; jc++) ccx[jc] = cx[2 * jc];
        for (int jc = 0; jc <= Mc; jc++) ccu[jc] = 2. / (1. / cu[2 * jc] + 1. / cu[2 * jc + 1]);
        cx.swap(ccx);
        cu.swap(ccu);
        N = Nc;
        M = Mc;
    }
    H.nlev = l;
    // exact solve of a small coarsest level: dense inverse of its operator
    // (SPD: diagonal 2 cx + cu_j + cu_{j-1}, -cx to the periodic x
    // neighbours, -cu to the z neighbours, Dirichlet rows dropped), by
    // Gauss-Jordan elimination in FP64
    {
        const int n = N * M;
        if (n > 0 && n <= 512) {
            std::vector<double> A(size_t(n) * n, 0.), I(size_t(n) * n, 0.);
            for (int j = 1; j <= M; j++)
                for (int i = 0; i < N; i++) {
                    const int t = (j - 1) * N + i;
                    A[size_t(t) * n + t] += 2. * cx[j] + cu[j] + cu[j - 1];
                    A[size_t(t) * n + (j - 1) * N + (i + N - 1) % N] -= cx[j];
                    A[size_t(t) * n + (j - 1) * N + (i + 1) % N] -= cx[j];
                    if (j + 1 <= M) A[size_t(t) * n + j * N + i] -= cu[j];
                    if (j - 1 >= 1) A[size_t(t) * n + (j - 2) * N + i] -= cu[j - 1];
                }
            for (int t = 0; t < n; t++) I[size_t(t) * n + t] = 1.;
            bool ok = true;
            for (int c = 0; c < n && ok; c++) {
                int piv = c;
                for (int r = c + 1; r < n; r++)
                    if (std::fabs(A[size_t(r) * n + c]) > std::fabs(A[size_t(piv) * n + c])) piv = r;
                if (A[size_t(piv) * n + c] == 0.) {
                    ok = false;
                    break;
                }
                if (piv != c)
                    for (int k = 0; k < n; k++) {
                        std::swap(A[size_t(c) * n + k], A[size_t(piv) * n + k]);
                        std::swap(I[size_t(c) * n + k], I[size_t(piv) * n + k]);
                    }
                const double inv = 1. / A[size_t(c) * n + c];
                for (int k = 0; k < n; k++) {
                    A[size_t(c) * n + k] *= inv;
                    I[size_t(c) * n + k] *= inv;
                }
                for (int r = 0; r < n; r++) {
                    if (r == c) continue;
                    const double fct = A[size_t(r) * n + c];
                    if (fct == 0.) continue;
                    for (int k = 0; k < n; k++) {
                        A[size_t(r) * n + k] -= fct * A[size_t(c) * n + k];
                        I[size_t(r) * n + k] -= fct * I[size_t(c) * n + k];
                    }
                }
            }
            if (ok) {
                std::vector<T> Ti(I.begin(), I.end());
                H.cinv = dalloc<T>(size_t(n) * n);
                if (!H.cinv) return false;
                hipMemcpy(H.cinv, Ti.data(), sizeof(T) * Ti.size(), hipMemcpyHostToDevice);
                H.cinv_n = n;
            }
        }
    }
    // the one-workgroup kernel takes every level that fits in 64 KiB of LDS;
    // the finest levels run as tiled down/up kernels
    return mg_plan(H, size_t(64) * 1024) == 0;
}

template <typename T>
void free_hier(MGHier<T> &H) {
    for (int l = 0; l < H.nlev; l++) {
        MGLevel<T> &L = H.lev[l];
        hipFree(L.cx);
        hipFree(L.cu);
        hipFree(L.dinv);
        if (l > 0) {
            hipFree(L.x);
            hipFree(L.b);
            hipFree(L.t);
        }
    }
    if (H.cws) hipFree(H.cws);
    H.cws = nullptr;
    if (H.cinv) hipFree(H.cinv);
    H.cinv = nullptr;
    H.cinv_n = 0;
    H.nlev = 0;
}

template <typename T>
bool pcg_fused(const PCG<T> &P, const RedSlot &rs, const double *hpart_dev) {
    return hpart_dev && mg_cg_fusable(P.mg, rs.max_blocks);
}

// The first V-cycle of pcg_loop (on P.r), which a caller may queue before it
// has read the initial residual, so that the GPU does not wait for the host;
// returns what pcg_loop's n_rz_pre takes.
template <typename T>
int pcg_first_vcycle(PCG<T> &P, const RedSlot &rs, const double *hpart_dev, hipStream_t st) {
    const bool fused = pcg_fused(P, rs, hpart_dev);
    // fused: r.z and w.z partials; otherwise r.z into sc[P_RZ]
    const int n = mg_vcycle(P.mg, P.r, P.zA, P.zB, rs, P.sc, true, st, false, fused ? P.w : nullptr);
    return fused ? n : 0;  // unfused: the first pq kernel takes beta = 0 and needs no partials
}

// Preconditioned CG iterations on P (x, r and sc[P_RNORM2] set up by the
// caller; rn_start = that ||w r||^2) until ||w r||^2 <= target or max_iter.
// The convergence test lags one V-cycle behind the GPU so the stream never
// drains: the next V-cycle is queued before the host reads the residual.
// When the residual history predicts that this iteration meets the target
// (geometric extrapolation of the last ratio), the V-cycle is queued only
// after the test, since a speculative V-cycle after the last iteration is
// wasted work; a wrong prediction costs one drained queue instead.  Returns
// the iteration count; *rn2 gets the last residual norm^2 seen.
//
// On a hierarchy with a tiled level 0 (every grid but the smallest) the
// iteration is the single-reduction form: the V-cycle's level-0 up kernel
// leaves r.z and w.z (w = L z), and the level-0 down kernel of the next
// V-cycle forms alpha and beta from them and applies the whole update, so an
// iteration is one V-cycle and nothing else.  Otherwise (a hierarchy that is
// only the coarse kernel) it is standard PCG with its own vector kernels.
template <typename T>
int pcg_loop(PCG<T> &P, double target, int max_iter, bool stall_stop, const RedSlot &rs, double *hs,
             double *hs_dev, const double *hpart, double *hpart_dev, hipEvent_t ev, hipStream_t st,
             double rn_start, double *rn2, bool *conv, int n_rz_pre = -1) {
    const bool fused = pcg_fused(P, rs, hpart_dev);
    const int nb = cg_blocks(P.N, P.M);
    const dim3 b(LX, LY);
    // p.q partials in the last row of the reduction slots, which the update
    // kernel reads while it writes its own partials to row 0
    const RedSlot rs_pq{rs.partial + size_t(7) * rs.max_blocks, rs.max_blocks};
    int n_rz = n_rz_pre >= 0 ? n_rz_pre : pcg_first_vcycle(P, rs, hpart_dev, st);
    int it = 0;
    double best = 1e300;
    int stall = 0;
    double prev = rn_start, prev2 = -1.;
    *conv = false;
    while (it < max_iter) {
        it++;
        const int rz_old = (it & 1) ? P_RZ2 : P_RZ, rz_now = (it & 1) ? P_RZ : P_RZ2;  // it = 1: P_RZ
        int nfused = 0;
        if (fused) {
            const int a_old = (it & 1) ? P_ALPHA2 : P_ALPHA, a_now = (it & 1) ? P_ALPHA : P_ALPHA2;
            const CGFuse<T> fz{P.x,  P.r,   P.rB,   P.pA,  P.q,         P.qB, P.w, P.wD, P.sc, rz_old,
                               rz_now, a_old, a_now, int(it == 1), rs, n_rz, hpart_dev};
            nfused = mg_down0_cg(P.mg, P.zA, fz, rs.max_blocks, st);
            std::swap(P.r, P.rB);
            std::swap(P.q, P.qB);
        } else {
            hipLaunchKernelGGL(k_pcg_pq<T>, dim3(nb), b, 0, st, P.N, P.M, P.zA, P.pA, P.pB, P.q, P.mg.lev[0].cx,
                               P.mg.lev[0].cu, P.sc, rs_pq, int(it == 1), rs, n_rz, rz_old, rz_now);
            std::swap(P.pA, P.pB);
            hipLaunchKernelGGL(k_pcg_update<T>, dim3(nb), b, 0, st, P.N, P.M, P.x, P.r, P.pA, P.q, P.wD, P.sc,
                               rz_now, rs_pq, nb, rs);
            finalize<1>(rs, nb, P.sc, RED_STORE, P_RNORM2, st, -1, hs_dev);
        }
        hipEventRecord(ev, st);
        bool ahead = it < max_iter;
        if (ahead && !stall_stop) {
            // an MG-PCG step cuts ||r||^2 by ~1e-2; the last observed ratio is a
            // better guess once there is one
            const double q = (prev2 > 0.) ? std::min(prev / prev2, 1.) : 1e-2;
            if (prev * q <= target) ahead = false;
        }
        T *wz = fused ? P.w : nullptr;
        if (ahead) n_rz = mg_vcycle(P.mg, P.r, P.zA, P.zB, rs, P.sc, false, st, fused, wz);
        hipEventSynchronize(ev);
        double rn = 0.;
        if (fused) {
            const volatile double *hp = hpart;
            for (int k = 0; k < nfused; k++) rn += hp[k];  // fixed order: deterministic
        } else {
            rn = *static_cast<volatile double *>(hs);
        }
        *rn2 = rn;
        if (!std::isfinite(rn)) break;  // breakdown (NaN or Inf): stop, not converged
        if (!(rn > target)) {
            *conv = true;
            break;
        }
        if (!ahead && it < max_iter) n_rz = mg_vcycle(P.mg, P.r, P.zA, P.zB, rs, P.sc, false, st, fused, wz);
        prev2 = prev;
        prev = rn;
        if (stall_stop) {
            if (rn < 0.25 * best) {
                best = rn;
                stall = 0;
            } else if (++stall >= 3) {
                *conv = true;
                break;
            }
        }
    }
    return it;
}

}  // namespace

int Poisson::init(const Grid &G, const double *rhou, const double *rhow, const RedSlot &rs, bool with_direct,
                  bool with_fp32, bool with_pcg) {
    N = G.nx - 2;
    M = G.nz - 3;
    red = rs;
    have_pcg = with_pcg;
    std::vector<double> cx(M + 2, 0.), cu(M + 1, 0.);
    for (int j = 1; j <= M; j++) cx[j] = 1. / rhow[j + 1];
    for (int j = 0; j <= M; j++) cu[j] = 1. / rhou[j + 1];
    const size_t n = size_t(M + 2) * N;
    std::vector<double> wd(M + 2, 0.);
    for (int j = 1; j <= M; j++) wd[j] = rhow[j + 1];
    cx0 = dalloc<double>(M + 2);
    cu0 = dalloc<double>(M + 1);
    if (!cx0 || !cu0) return VVM_ERR_NOMEM;
    hipMemcpy(cx0, cx.data(), sizeof(double) * (M + 2), hipMemcpyHostToDevice);
    hipMemcpy(cu0, cu.data(), sizeof(double) * (M + 1), hipMemcpyHostToDevice);
    PCG<double> &P = pcg64;
    P.N = N;
    P.M = M;
    P.x = dalloc<double>(n);
    P.r = dalloc<double>(n);
    P.wD = dalloc<double>(M + 2);
    P.sc = dalloc<double>(NPSCAL);
    if (!P.x || !P.r || !P.wD || !P.sc) return VVM_ERR_NOMEM;
    hipMemcpy(P.wD, wd.data(), sizeof(double) * (M + 2), hipMemcpyHostToDevice);
    if (with_pcg) {
        if (!build_hier(P.mg, N, M, cx, cu)) return VVM_ERR_NOMEM;
        for (double **v : {&P.rB, &P.zA, &P.zB, &P.pA, &P.pB, &P.q, &P.qB, &P.w})
            if (!(*v = dalloc<double>(n))) return VVM_ERR_NOMEM;
    }
    if (with_direct)
        if (const int rc = direct64.init(N, M, cx0, cu0)) return rc;
    if (with_fp32)
        if (const int rc = direct32.init(N, M, cx0, cu0)) return rc;
    f = dalloc<double>(n);
    xprev = dalloc<double>(n);
    xprev2 = dalloc<double>(n);
    xprev3 = dalloc<double>(n);
    x64B = dalloc<double>(n);
    if (!f || !xprev || !xprev2 || !xprev3 || !x64B) return VVM_ERR_NOMEM;
    // pinned, coherent and mapped: k_finalize writes the CG residual norm
    // here directly, and the host reads it after an event
    if (hipHostMalloc(reinterpret_cast<void **>(&hscal), 16 * sizeof(double),
                      hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess)
        return VVM_ERR_NOMEM;
    if (hipHostGetDevicePointer(reinterpret_cast<void **>(&hscal_dev), hscal, 0) != hipSuccess) return VVM_ERR_HIP;
    if (hipHostMalloc(reinterpret_cast<void **>(&hres), 4 * kResidualBlocks * sizeof(double),
                      hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess)
        return VVM_ERR_NOMEM;
    if (hipHostGetDevicePointer(reinterpret_cast<void **>(&hres_dev), hres, 0) != hipSuccess) return VVM_ERR_HIP;
    // per-workgroup residual norms of the fused CG update, read by the host
    if (hipHostMalloc(reinterpret_cast<void **>(&hpart), sizeof(double) * size_t(rs.max_blocks),
                      hipHostMallocMapped | hipHostMallocCoherent) != hipSuccess)
        return VVM_ERR_NOMEM;
    if (hipHostGetDevicePointer(reinterpret_cast<void **>(&hpart_dev), hpart, 0) != hipSuccess) return VVM_ERR_HIP;
    if (hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess) return VVM_ERR_HIP;
    if (hipEventCreateWithFlags(&ev_res, hipEventDisableTiming) != hipSuccess) return VVM_ERR_HIP;
    // the zeroing of the allocations, before anything on the caller's stream
    return hipStreamSynchronize(nullptr) == hipSuccess ? VVM_OK : VVM_ERR_HIP;
}

template <typename T>
static void free_pcg(PCG<T> &P) {
    free_hier(P.mg);
    for (void *p : {(void *)P.x, (void *)P.r, (void *)P.rB, (void *)P.zA, (void *)P.zB, (void *)P.pA,
                    (void *)P.pB, (void *)P.q, (void *)P.qB, (void *)P.w, (void *)P.wD, (void *)P.sc})
        if (p) hipFree(p);
    P = PCG<T>();
}

void Poisson::destroy() {
    free_pcg(pcg64);
    have_pcg = false;
    direct64.destroy();
    direct32.destroy();
    for (void *p : {(void *)f, (void *)xprev, (void *)xprev2, (void *)xprev3, (void *)x64B, (void *)bcg, (void *)bsc,
                    (void *)cx0, (void *)cu0, (void *)gfeat, (void *)gsc, (void *)samples})
        if (p) hipFree(p);
    f = xprev = xprev2 = xprev3 = x64B = bcg = bsc = cx0 = cu0 = nullptr;
    gfeat = samples = nullptr;
    bn_pending = 0;
    x_pending = 0;
    if (hres) hipHostFree(hres);
    hres = hres_dev = nullptr;
    gsc = nullptr;
    gscratch.release();
    sample_cap = sample_count = 0;
    net = nullptr;
    if (hscal) hipHostFree(hscal);
    hscal = nullptr;
    hscal_dev = nullptr;
    if (hpart) hipHostFree(hpart);
    hpart = hpart_dev = nullptr;
    if (ev) hipEventDestroy(ev);
    if (ev_res) hipEventDestroy(ev_res);
    ev_res = nullptr;
    ev = nullptr;
}

int Poisson::replan(size_t budget) {
    if (budget > size_t(64) * 1024) return VVM_ERR_ARG;
    if (have_pcg && mg_plan(pcg64.mg, budget) != 0) return VVM_ERR_NOMEM;
    lds_budget = budget;
    return VVM_OK;
}

// ||b||^2 partials go to row 1 of red; the first residual's reduction adds
// them up with its own (flush_pending, if something needs red first)
void Poisson::rhs_from_zetap(const Grid &G, const double *zetap, const double *rhow_dev, hipStream_t st) {
    const RedSlot row1{red.partial + red.max_blocks, red.max_blocks};
    hipLaunchKernelGGL(k_calw_rhs, lgrid(N, M), dim3(LX, LY), 0, st, G, zetap, rhow_dev, f, pcg64.sc, row1);
    bn_pending = nblocks(lgrid(N, M));
}

void Poisson::rhs_from_b(const double *b, hipStream_t st) {
    // the FP64 row weights wD[j] are rhow[j+1]
    const RedSlot row1{red.partial + red.max_blocks, red.max_blocks};
    hipLaunchKernelGGL(k_rhs_from_b, lgrid(N, M), dim3(LX, LY), 0, st, N, M, b, pcg64.wD, f, pcg64.sc, row1);
    bn_pending = nblocks(lgrid(N, M));
}

void Poisson::flush_pending(hipStream_t st) {
    if (bn_pending) {
        const RedSlot row1{red.partial + red.max_blocks, red.max_blocks};
        finalize<1>(row1, bn_pending, pcg64.sc, RED_STORE, P_BNORM2, st, -1, hscal_dev + P_BNORM2);
        bn_pending = 0;
    }
    const size_t n = size_t(M + 2) * N;
    if (x_pending == XF_ZERO)
        hipMemsetAsync(pcg64.x, 0, n * sizeof(double), st);
    else if (x_pending == XF_EXTRAP)
        hipLaunchKernelGGL(k_extrapolate, dim3((n + 255) / 256), dim3(256), 0, st, n, pcg64.x, xprev, xprev2, xprev3,
                           x_pending_ord);
    x_pending = XF_NONE;
}

void Poisson::first_residual(double *r, hipStream_t st) {
    const dim3 g = lgrid(N, M), b(LX, LY);
    PCG<double> &D = pcg64;
#define VVM_RESIDUAL_X(XF)                                                                                         \
    hipLaunchKernelGGL((k_residual_x<XF>), g, b, 0, st, N, M, f, D.x, xprev, xprev2, xprev3, x_pending_ord, r, cx0, \
                       cu0, D.wD, red)
    switch (x_pending) {
        case XF_EXTRAP: VVM_RESIDUAL_X(XF_EXTRAP); break;
        case XF_ZERO: VVM_RESIDUAL_X(XF_ZERO); break;
        default: VVM_RESIDUAL_X(XF_NONE); break;
    }
#undef VVM_RESIDUAL_X
    x_pending = XF_NONE;
    // the norms land in mapped host memory (hscal) directly: no copy in the stream
    if (bn_pending) {
        // rows 0 (r) and 1 (b), same grid: sc[P_RNORM2], sc[P_BNORM2]
        finalize<2>(red, nblocks(g), D.sc, RED_STORE, P_RNORM2, st, -1, hscal_dev + P_RNORM2);
        bn_pending = 0;
    } else {
        finalize<1>(red, nblocks(g), D.sc, RED_STORE, P_RNORM2, st, -1, hscal_dev + P_RNORM2);
    }
}

void Poisson::x_to_ref(double *xref, hipStream_t st) {
    hipLaunchKernelGGL(k_x_ref, lgrid(N, M), dim3(LX, LY), 0, st, N, M, pcg64.x, xref, 1);
}

void Poisson::x_from_ref(const double *xref, hipStream_t st) {
    hipLaunchKernelGGL(k_x_ref, lgrid(N, M), dim3(LX, LY), 0, st, N, M, pcg64.x, const_cast<double *>(xref), 0);
}

void Poisson::back_to_w(const Grid &G, double *w, const double *rhow_dev, hipStream_t st) {
    hipLaunchKernelGGL(k_calw_back, dim3((G.nx + LX - 1) / LX, (G.nz + LY - 1) / LY), dim3(LX, LY), 0, st, G, pcg64.x,
                       w, rhow_dev);
}

void Poisson::set_guess(int mode, hipStream_t st) {
    guess_from_net = false;
    // formed by the solve's first residual kernel (first_residual)
    x_pending = XF_NONE;
    if (mode == VVM_GUESS_ZERO) {
        x_pending = XF_ZERO;
    } else if ((mode == VVM_GUESS_EXTRAP || mode == VVM_GUESS_EXTRAP2) && nsolves >= 2) {
        x_pending = XF_EXTRAP;
        x_pending_ord = (mode == VVM_GUESS_EXTRAP2) ? xe_order() : 1;
    }
    // VVM_GUESS_PREV, and the extrapolations before two solutions exist,
    // start from the last solution (x holds the oldest one after
    // remember_solution); the learned guess is written by its own kernels.
    if (x_pending == XF_NONE && mode != VVM_GUESS_ZERO && nsolves >= 1)
        hipMemcpyAsync(pcg64.x, xprev, size_t(M + 2) * N * sizeof(double), hipMemcpyDeviceToDevice, st);
}

void Poisson::remember_solution(hipStream_t st) {
    flush_pending(st);  // nothing is pending after a solve; a guess set without one is formed now
    // x_{t-3} <- x_{t-2} <- x_{t-1} <- x by rotating the buffers, no copy:
    // the oldest becomes the next solve's x, which set_guess fills (or the
    // first residual kernel, or the network, rewrites in full)
    double *oldest = xprev3;
    xprev3 = xprev2;
    xprev2 = xprev;
    xprev = pcg64.x;
    pcg64.x = oldest;
    nsolves++;
}

// Whether the solve keeps the network's guess, whose residual is rn2.
bool Poisson::keep_guess(double rn2) {
    if (std::isfinite(rn2) && rn2 <= hscal[H_GUESS + 3]) {
        net_backoff = 0;
        return true;
    }
    net_backoff = std::min(std::max(1, 4 * net_backoff), kMaxNetSkip);
    net_skip = net_backoff;
    guess_fallbacks++;
    return false;
}

void Poisson::start_solve(double *r, int *n_rz_pre, double *bn2, double *rn2, hipStream_t st) {
    const bool judge = guess_from_net;
    guess_from_net = false;
    for (int attempt = 0;; attempt++) {
        first_residual(r, st);
        hipEventRecord(ev_res, st);
        *n_rz_pre = pcg_first_vcycle(pcg64, red, hpart_dev, st);
        hipEventSynchronize(ev_res);
        *bn2 = hscal[P_BNORM2];
        *rn2 = hscal[P_RNORM2];
        if (!judge || attempt > 0 || keep_guess(*rn2)) return;
        // the network's guess starts worse than the extrapolation it corrects
        // (or is not finite): start from the extrapolation instead; the first
        // V-cycle queued on the rejected residual is simply overwritten
        x_pending = XF_EXTRAP;
        x_pending_ord = xe_order();
    }
}

SolveResult Poisson::solve_fp64(double tol, int max_iter, hipStream_t st) {
    SolveResult R;
    PCG<double> &P = pcg64;
    // the first V-cycle goes in before the host reads the residual (a guess
    // that already meets the stop rule wastes it, which is rare)
    int n_rz_pre = 0;
    double bn2 = 0., rn2 = 0.;
    start_solve(P.r, &n_rz_pre, &bn2, &rn2, st);
    if (!std::isfinite(bn2) || !std::isfinite(rn2)) {  // a non-finite right-hand side or guess
        R.rel0 = R.rel = std::sqrt(rn2 / bn2);
        return R;
    }
    if (bn2 == 0.) {
        hipMemsetAsync(P.x, 0, size_t(M + 2) * N * sizeof(double), st);
        R.converged = true;
        return R;
    }
    R.rel0 = std::sqrt(rn2 / bn2);
    const bool parity = (tol <= 0.);
    const double target = parity ? 1e-30 * bn2 : tol * tol * bn2;
    if (!(rn2 > target)) {
        R.rel = R.rel0;
        R.converged = true;
        return R;
    }
    double last = rn2;
    bool conv = false;
    R.iters = pcg_loop(P, target, max_iter, parity, red, hscal + 8, hscal_dev + 8, hpart, hpart_dev, ev, st, rn2, &last,
                       &conv, n_rz_pre);
    R.rel = std::sqrt(last / bn2);
    R.converged = conv;
    return R;
}

// Relative residual up to which one that no longer decreases counts as FP64's
// round-off: 2^-53 times the largest condition number, 8 (M + 1)^2 / pi^2 times
// the density's range over the column, 4e-10 at 480 levels.  2^-53 of ||L|| ||x|| is 1e-16 of
// ||b|| where b is rough, 3e-14 on k^-3 vorticity and 1e-12 on the lowest mode
// (2048 x 256).  One solve leaves three to five times that and an error of up
// to 3e-14, and a correction cuts an error by at least 1e-9, so that the
// second solve always reaches the floor: 512 x 64, k^-3 vorticity, one / two /
// three solves leave residuals of 4.6e-14 / 1.1e-14 / 1.1e-14 and errors of
// 1.2e-14 / 9e-17 / 9e-17.
constexpr double kRoundOff = 1e-9;

// Norms of the residual kernel's slot (the caller has waited for it).
void Poisson::norms(int slot, double *rn2, double *bn2) const {
    const volatile double *p = slot_host(slot);
    *rn2 = *bn2 = 0.;
    for (int b = 0; b < res_blocks; b++) {  // fixed order: deterministic
        *rn2 += p[2 * b];
        *bn2 += p[2 * b + 1];
    }
}

// r of x (with ref: of the given right-hand side and guess), norms into slot.
void Poisson::queue_r(const RefArrays *ref, int slot, hipStream_t st) {
    res_blocks = residual_blocks();
    const Residual R{N, M, f, pcg64.x, cx0, cu0, pcg64.wD, slot_dev(slot)};
    if (ref)
        hipLaunchKernelGGL(k_solve_residual<true>, dim3(res_blocks), dim3(1024), 0, st, R, ref->b, ref->x, f,
                           pcg64.x, pcg64.r);
    else
        hipLaunchKernelGGL(k_solve_residual<false>, dim3(res_blocks), dim3(1024), 0, st, R, nullptr, nullptr, nullptr,
                           nullptr, pcg64.r);
}

// Whether a correction that took the relative residual from prev to R.rel was
// the last, and (R.converged) met the stop rule.
static bool at_end(SolveResult &R, double prev, double tol, Floor floor) {
    const bool stalled = R.rel > 0.5 * prev;
    R.converged = R.rel <= tol || (floor != Floor::NONE && stalled && R.rel <= kRoundOff) ||
                  (floor == Floor::PARITY && prev <= kRoundOff);
    return R.converged || stalled;
}

// Each sweep: x += L^-1 r by a direct solve, formed in another buffer, the FP64
// residual and (ref) the solution in the reference's order, all queued before
// the host reads the norms; the first sweep also before it has read those of
// the guess, which may already meet the stop rule.  2048 x 255 in FP64, two
// sweeps: 120 us, 11 launches and two waits.
template <typename T>
SolveResult Poisson::refine(Direct<T> &D, const RefArrays *ref, double tol, Floor floor, int max_sweeps,
                            hipStream_t st) {
    SolveResult R;
    double rn2 = 0., bn2 = 0.;
    auto out = [&] {
        if (!ref) return;
        hipEventRecord(ref->done, st);
        x_to_ref(ref->x, st);
    };
    auto correct = [&] {
        D.solve(pcg64.r, pcg64.x, x64B, st);
        std::swap(pcg64.x, x64B);
        queue_r(nullptr, 1, st);
        out();
        hipStreamSynchronize(st);
    };
    x_pending = XF_NONE;
    queue_r(ref, 0, st);
    correct();
    norms(0, &rn2, &bn2);
    const bool finite = std::isfinite(bn2) && std::isfinite(rn2);  // else: a bad right-hand side or guess
    R.rel = R.rel0 = std::sqrt(rn2 / bn2);
    R.converged = finite && (bn2 == 0. || R.rel <= tol);
    if (R.converged || !finite || max_sweeps < 1) {  // the guess stays
        if (finite && bn2 == 0.) {
            R = SolveResult();
            R.converged = true;
            hipMemsetAsync(x64B, 0, size_t(M + 2) * N * sizeof(double), st);
        }
        std::swap(pcg64.x, x64B);
        out();
        return R;
    }
    for (int sweep = 1;; sweep++) {
        const double prev = R.rel;
        norms(1, &rn2, &bn2);
        R.rel = std::sqrt(rn2 / bn2);
        R.iters = R.refine = sweep;
        if (!std::isfinite(bn2) || !std::isfinite(rn2)) return R;
        if (at_end(R, prev, tol, floor) || sweep == max_sweeps) return R;
        correct();
    }
}

SolveResult Poisson::solve_direct(const RefArrays &ref, double tol, Floor floor, int max_sweeps, hipStream_t st) {
    SolveResult R = refine(direct64, &ref, tol, floor, max_sweeps, st);
    R.refine = 0;
    return R;
}

SolveResult Poisson::solve_mixed(const RefArrays &ref, double tol, int max_sweeps, hipStream_t st) {
    return refine(direct32, &ref, tol, Floor::NONE, max_sweeps, st);
}

void Poisson::queue_step(const Grid &G, const StepPtrs &S, int step, bool f_ready, const Micro *micro,
                         hipStream_t st) {
    double *w = S.w;
    const double *rhow_dev = S.P.rhow;
    x_pending = XF_NONE;
    if (step >= 0 && (guess_from_net || f_ready)) launch_pubartop(G, S, step, st);
    if (guess_from_net) {
        guess_from_net = false;
        first_residual(pcg64.r, st);
        hipEventRecord(ev_res, st);
        hipEventSynchronize(ev_res);
        if (keep_guess(hscal[P_RNORM2])) {
            direct64.solve(pcg64.r, pcg64.x, x64B, st);
            std::swap(pcg64.x, x64B);
        } else {
            direct64.solve(f, nullptr, pcg64.x, st);
        }
        back_to_w(G, w, rhow_dev, st);
    } else if (f_ready) {
        direct64.solve(f, nullptr, pcg64.x, st);
        back_to_w(G, w, rhow_dev, st);
    } else {
        direct64.solve_step(G, S, step, micro, f, pcg64.x, st);
    }
    bn_pending = 0;
    corrected = expect_more;
    if (corrected) {
        mark_unset(slot_host(0), 2 * residual_blocks());
        queue_r(nullptr, 0, st);
        direct64.solve_w(pcg64.r, pcg64.x, x64B, G, w, rhow_dev, st);
        std::swap(pcg64.x, x64B);
    }
}

SolveResult Poisson::finish_step(const Grid &G, double *w, const double *rhow_dev, double tol, Floor floor,
                                 int max_sweeps, bool *redo, hipStream_t st) {
    SolveResult R;
    *redo = false;
    double rn2 = 0., bn2 = 0.;
    const bool more = corrected;
    corrected = expect_more = false;
    await_set(slot_host(0), 2 * res_blocks, st);
    if (more) await_set(slot_host(1), 2 * res_blocks, st);
    norms(0, &rn2, &bn2);
    R.iters = 1;
    R.rel0 = 1.;
    R.rel = bn2 > 0. ? std::sqrt(rn2 / bn2) : std::sqrt(rn2);
    R.converged = std::isfinite(bn2) && R.rel <= tol;
    if (R.converged || !std::isfinite(R.rel) || max_sweeps <= 1) {
        if (more) {
            hipStreamSynchronize(st);  // what is queued again marks its sums unset
            std::swap(pcg64.x, x64B);
            back_to_w(G, w, rhow_dev, st);
            *redo = true;
        }
        return R;
    }
    // beyond what one solve gives: corrected further
    expect_more = true;
    if (more) {
        const double prev = R.rel;
        norms(1, &rn2, &bn2);
        R.rel = std::sqrt(rn2 / bn2);
        R.iters = 2;
        R.refine = 1;
        if (!std::isfinite(R.rel) || at_end(R, prev, tol, floor) || max_sweeps <= 2) return R;
    }
    SolveResult C = refine(direct64, nullptr, tol, floor, max_sweeps - R.iters, st);
    C.iters += R.iters;
    C.refine += R.refine;
    C.rel0 = 1.;
    back_to_w(G, w, rhow_dev, st);
    *redo = true;
    return C;
}

// ---------------------------------------------------------------- cal_u

bool cal_u_supported(const Grid &G) { return G.nx - 2 <= 8192; }

void launch_cal_u(const Grid &G, const StepPtrs &S, hipStream_t st) {
    const int N = G.nx - 2, ncol = (N + UW - 1) / UW;
    hipLaunchKernelGGL(k_calu, dim3(ncol), dim3(UW * UC), size_t(N) * sizeof(double), st, G, S, ncol, Residual{});
}

void Poisson::queue_cal_u(const Grid &G, const StepPtrs &S, hipStream_t st) {
    const int ncol = (N + UW - 1) / UW;
    queue_residual(G, S, ncol, st);
}

void Poisson::queue_check(hipStream_t st) { queue_residual(Grid{}, StepPtrs{}, 0, st); }

// k_calu's residual workgroups, behind ncol workgroups of cal_u
void Poisson::queue_residual(const Grid &G, const StepPtrs &S, int ncol, hipStream_t st) {
    res_blocks = residual_blocks();
    const int slot = corrected ? 1 : 0;
    mark_unset(slot_host(slot), 2 * res_blocks);
    hipLaunchKernelGGL(k_calu, dim3(ncol + res_blocks), dim3(UW * UC), ncol ? size_t(N) * sizeof(double) : 0, st, G,
                       S, ncol, Residual{N, M, f, pcg64.x, cx0, cu0, pcg64.wD, slot_dev(slot)});
}

}  // namespace vvmd
