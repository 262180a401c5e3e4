// k_physics.hip -- Kessler microphysics, first-order turbulence closure and
// K-diffusion, nudging and horizontal means of one VVM timestep (phases C-E
// of vvm::Iteration::TimeMarching, src/Iteration.cpp:300-434).
//
// FP64, no FMA contraction (reference rounding, see k_dynamics.hip).
// std::max(a,b) / std::min(a,b) keep their NaN behaviour: (a<b)?b:a and
// (b<a)?b:a.
#pragma clang fp contract(off)

#include "micro.h"
#include "vvm_internal.h"

#include <cstdio>
#include <mutex>

namespace vvmd {

namespace {

constexpr int BX = 64, BY = 4;

__device__ inline double max_or_nan(double a, double b) { return (a != a || a > b) ? a : b; }

inline dim3 grid2d(const Grid &G) { return dim3((G.nx + BX - 1) / BX, (G.nz + BY - 1) / BY); }
// from the first interior point on: one tile less where the grid's columns and
// rows are multiples of the tile, and with it the last, nearly empty round
inline dim3 interior_grid(const Grid &G) { return dim3((G.nx - 2 + BX - 1) / BX, (G.nz - 2 + BY - 1) / BY); }

template <int PROC>
__global__ void __launch_bounds__(BX *BY) k_kessler(Grid G, StepPtrs S, Negval nv, Forcing F, RedSlot rs) {
    const int i = 1 + blockIdx.x * BX + threadIdx.x, k = 1 + blockIdx.y * BY + uniform(threadIdx.y);
    double part[6] = {0., 0., 0., 0., 0., 0.};
    double ratios[3] = {-1., -1., -1.};
    if constexpr ((PROC & KP_PRE) != 0) {
        note_start(S.clock, CLK_MICRO);
        negval_ratios(S, nv.rs, nv.nblk, ratios);
    }
    if (i <= G.nx - 2 && k <= G.nz - 2) kessler_point<PROC>(G, S, F, ratios, i, k, part);
    if constexpr ((PROC & KP_NEG) != 0) block_partials<6>(part, rs);
}

// MicroPhysics::NegativeValueProcess (MicroPhysics.cpp:116-138) on one
// field: the first pass zeroes the negatives and sums positives and
// negatives (k_finalize forms the ratio), the second rescales.
__global__ void __launch_bounds__(BX *BY) k_negval_sums(Grid G, double *a, RedSlot rs) {
    const int i = blockIdx.x * BX + threadIdx.x, k = blockIdx.y * BY + uniform(threadIdx.y);
    double part[2] = {0., 0.};
    if (i >= 1 && i <= G.nx - 2 && k >= 1 && k <= G.nz - 2) {
        const double v = at(a, G, i, k);
        if (v >= 0.) part[0] += v;
        else {
            part[1] += v;
            at(a, G, i, k) = 0.;
        }
    }
    block_partials<2>(part, rs);
}
__global__ void __launch_bounds__(BX *BY) k_negval_scale(Grid G, double *a, const double *ratio) {
    const int i = blockIdx.x * BX + threadIdx.x, k = blockIdx.y * BY + uniform(threadIdx.y);
    if (i < 1 || i > G.nx - 2 || k < 1 || k > G.nz - 2) return;
    const double r = *ratio;
    if (r >= 0. && at(a, G, i, k) > 0) at(a, G, i, k) = at(a, G, i, k) * r;
}

// Turbulence::RKM_RKH coefficient part (Turbulent.cpp:13-45), with the
// center halos of RKM and RKH.  Returns the larger of the two, and NaN where th
// is not finite (ALL: any field that is diffused, or a neighbour of it): such a
// value reaches every point to its east and above, so the sweep has to run in
// order.  The coefficients do not tell: a Richardson number that is NaN gives
// the smallest.  In a step without host microphysics th is enough: zeta shows in the solve's residual, and
// the microphysics' negative-value pass leaves no such qv, qc or qr.
template <bool ALL>
__device__ inline double turb_point(const Grid &G, const StepPtrs &S, int i, int k) {
    const double *u = S.u, *w = S.w, *thp = S.fut[F_TH];
    const double Rz =
        0.5 * ((at(w, G, i + 1, k + 1) + at(w, G, i + 1, k)) - (at(w, G, i - 1, k + 1) + at(w, G, i - 1, k))) * G.r2dx +
        0.5 * ((at(u, G, i + 1, k + 1) + at(u, G, i, k + 1)) - (at(u, G, i + 1, k - 1) + at(u, G, i, k - 1))) * G.r2dz;
    const double dv = (at(u, G, i + 1, k) - at(u, G, i, k)) * G.rdx + (at(w, G, i, k + 1) - at(w, G, i, k)) * G.rdz;
    const double Ro = dv * dv;
    const double Ri = (G.GRAVITY / at(thp, G, i, k) * (at(thp, G, i, k + 1) - at(thp, G, i, k - 1)) * G.r2dz) /
                      (Rz * Rz + 2. * Ro);
    const double l2 = S.P.lambda2[k];
    double km, kh;
    if (Ri < 0) {
        km = l2 * sqrt(Rz * Rz + 2. * Ro) * sqrt(1. - 16. * Ri);
        kh = l2 * sqrt(Rz * Rz + 2. * Ro) * 1.4 * sqrt(1. - 40. * Ri);
    } else if (0 < Ri && Ri < 0.25) {
        km = l2 * sqrt(Rz * Rz + 2. * Ro) * pow(1. - 4. * Ri, 4.);
        kh = l2 * sqrt(Rz * Rz + 2. * Ro) * 1.4 * (1. - 1.2 * Ri) * pow(1. - 4. * Ri, 4.);
    } else {
        km = 0.;
        kh = 0.;
    }
    const double kmax = 0.8 * G.dx * G.dz / G.dt;
    km = maxs(km, 10.);
    kh = maxs(kh, 10.);
    km = mins(km, kmax);
    kh = mins(kh, kmax);
    store_center(S.RKM, G, i, k, km);
    store_center(S.RKH, G, i, k, kh);
    bool finite = __builtin_isfinite(at(thp, G, i, k));
    if constexpr (ALL) {
        for (const double *f : S.fut)
            for (double v : {at(f, G, i, k), at(f, G, i - 1, k), at(f, G, i + 1, k), at(f, G, i, k - 1),
                             at(f, G, i, k + 1)})
                finite = finite && __builtin_isfinite(v);
    }
    return finite ? max_or_nan(km, kh) : __builtin_nan("");
}

constexpr int TBY = 16;
// At most kTurbBlocks workgroups walk the tiles (few and large: every one ends
// with a store to host memory, and 1089 of them made the kernel 2 us longer); each leaves the largest
// coefficient it formed in kmax, from which the host chooses the diffusion
// sweep.  A NaN (unstable stratification at rest: Ri = -inf; fields that are not
// finite) stays one.
template <bool ALL>
__global__ void __launch_bounds__(BX *TBY) k_turb_coeffs(Grid G, StepPtrs S, double *kmax) {
    note_start(S.clock, CLK_TURB);
    const int tx = (G.nx - 2 + BX - 1) / BX, nt = tx * ((G.nz - 2 + TBY - 1) / TBY);
    double m = 0.;
    for (int t = blockIdx.x; t < nt; t += gridDim.x) {
        const int i = 1 + (t % tx) * BX + threadIdx.x, k = 1 + (t / tx) * TBY + uniform(threadIdx.y);
        if (i < 1 || i > G.nx - 2 || k < 1 || k > G.nz - 2) continue;
        const double v = turb_point<ALL>(G, S, i, k);
        m = max_or_nan(m, v);
    }
    // m >= 0 or NaN, so that a lane without a partner takes 0 (dpp)
    m = max_or_nan(m, dpp<DPP_ROW_SHR + 1>(m));
    m = max_or_nan(m, dpp<DPP_ROW_SHR + 2>(m));
    m = max_or_nan(m, dpp<DPP_ROW_SHR + 4>(m));
    m = max_or_nan(m, dpp<DPP_ROW_SHR + 8>(m));
    m = max_or_nan(m, dpp<DPP_ROW_BCAST15, 0xa>(m));
    m = max_or_nan(m, dpp<DPP_ROW_BCAST31, 0xc>(m));
    __shared__ double sh[TBY];
    if (threadIdx.x == kWave - 1) sh[threadIdx.y] = m;
    __syncthreads();
    if (threadIdx.x == 0 && threadIdx.y == 0) {
        m = sh[0];
        for (int w = 1; w < TBY; w++) m = max_or_nan(m, sh[w]);
        __hip_atomic_store(kmax + blockIdx.x, m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}


// NumericalProcess::Nudge_qv (NumericalProcess.cpp:86-95), all points.
__global__ void __launch_bounds__(BX *BY) k_nudge_qv(Grid G, StepPtrs S, double tau) {
    const int i = blockIdx.x * BX + threadIdx.x, k = blockIdx.y * BY + threadIdx.y;
    if (i >= G.nx || k >= G.nz) return;
    const size_t p = ix(G, i, k);
    S.fut[F_QV][p] = S.fut[F_QV][p] + G.dt * (S.P.qvb0[k] - S.now[F_QV][p]) / tau;
}

// Iteration::updateMean (src/Iteration.cpp:42-86) as called by
// nextTimeStep: one block per level.  thb_zeta is not read by the step and
// is formed on download.
__global__ void __launch_bounds__(256) k_update_mean(Grid G, StepPtrs S, MeanMode mode) {
    note_start(S.clock, CLK_MEAN);
    const int k = blockIdx.x + 1;
    const double *thp = S.fut[F_TH], *qvp = S.fut[F_QV];
    double acc[2] = {0., 0.};
    for (int i = 1 + threadIdx.x; i < G.nx - 1; i += blockDim.x) {
        acc[0] += thp[ix(G, i, k)];
        acc[1] += qvp[ix(G, i, k)];
    }
    block_sum<2>(acc);
    if (threadIdx.x == 0) {
        double *thb = S.P.thb, *qvb = S.P.qvb, *thvb = S.P.thvb;
        const double tb = acc[0] / (double)(G.nx - 2.), qb = acc[1] / (double)(G.nx - 2.);
        const double tv = tb * (1 + 0.608 * qb);
        const bool shift = mode != MEAN_AGAIN;
        if (shift) S.P.thbm[k] = thb[k];
        if (shift) S.P.thvbm[k] = thvb[k];
        thb[k] = tb;
        qvb[k] = qb;
        thvb[k] = tv;
        if (k == 1) {
            if (shift) S.P.thbm[0] = thb[0];
            if (shift) S.P.thvbm[0] = thvb[0];
            thb[0] = tb;
            qvb[0] = qb;
            thvb[0] = tv;
            if (mode == MEAN_STEP) {
                // nextTimeStep's copy loop (src/Iteration.cpp:166-167)
                S.s[S_UBARTOPM] = S.s[S_UBARTOPP];
                S.s[S_UBARTOP] = S.s[S_UBARTOPP];
            }
        }
        if (k == G.nz - 2) {
            if (shift) S.P.thbm[k + 1] = thb[k + 1];
            if (shift) S.P.thvbm[k + 1] = thvb[k + 1];
            thb[k + 1] = tb;
            qvb[k + 1] = qb;
            thvb[k + 1] = tv;
        }
    }
}

}  // namespace

Negval launch_kessler(const Grid &G, const StepPtrs &S, const RedSlot &rs, hipStream_t st) {
    hipLaunchKernelGGL(k_kessler<KP_ALL>, interior_grid(G), dim3(BX, BY), 0, st, G, S, Negval{}, Forcing{}, rs);
    return {rs, nblocks(interior_grid(G))};
}
Negval launch_kessler(const Grid &G, const StepPtrs &S, const Negval &nv, const Forcing &F, const RedSlot &rs,
                      hipStream_t st) {
    if (past_caches(G))
        hipLaunchKernelGGL((k_kessler<KP_ALL | KP_PRE | KP_PAST>), interior_grid(G), dim3(BX, BY), 0, st, G, S, nv, F, rs);
    else
        hipLaunchKernelGGL((k_kessler<KP_ALL | KP_PRE>), interior_grid(G), dim3(BX, BY), 0, st, G, S, nv, F, rs);
    return {rs, nblocks(interior_grid(G))};
}
void launch_kessler_process(const Grid &G, const StepPtrs &S, int process, hipStream_t st) {
    const RedSlot none{nullptr, 0};
    switch (process) {
        case 0: hipLaunchKernelGGL(k_kessler<KP_AUTO>, interior_grid(G), dim3(BX, BY), 0, st, G, S, Negval{}, Forcing{}, none); break;
        case 1: hipLaunchKernelGGL(k_kessler<KP_ACCR>, interior_grid(G), dim3(BX, BY), 0, st, G, S, Negval{}, Forcing{}, none); break;
        case 2: hipLaunchKernelGGL(k_kessler<KP_EVAP>, interior_grid(G), dim3(BX, BY), 0, st, G, S, Negval{}, Forcing{}, none); break;
        default: hipLaunchKernelGGL(k_kessler<KP_COND>, interior_grid(G), dim3(BX, BY), 0, st, G, S, Negval{}, Forcing{}, none); break;
    }
}
void launch_negative_value(const Grid &G, const StepPtrs &S, double *a, const RedSlot &rs, hipStream_t st) {
    hipLaunchKernelGGL(k_negval_sums, grid2d(G), dim3(BX, BY), 0, st, G, a, rs);
    finalize<2>(rs, nblocks(grid2d(G)), S.s, RED_NEGVAL, S_NEG_RATIO, st);
    hipLaunchKernelGGL(k_negval_scale, grid2d(G), dim3(BX, BY), 0, st, G, a, S.s + S_NEG_RATIO);
}
int launch_turbulence_coeffs(const Grid &G, const StepPtrs &S, double *kmax, bool all, hipStream_t st) {
    const int nt = ((G.nx - 2 + BX - 1) / BX) * ((G.nz - 2 + TBY - 1) / TBY), turns = (nt + kTurbBlocks - 1) / kTurbBlocks,
              nb = (nt + turns - 1) / turns;
    if (all) hipLaunchKernelGGL(k_turb_coeffs<true>, dim3(nb), dim3(BX, TBY), 0, st, G, S, kmax);
    else hipLaunchKernelGGL(k_turb_coeffs<false>, dim3(nb), dim3(BX, TBY), 0, st, G, S, kmax);
    return nb;
}

// Nudge_theta and Nudge_zeta alone (NumericalProcess.cpp:60-84), pointwise;
// the timestep fuses them into the diffusion sweep instead.
__global__ void __launch_bounds__(BX *BY) k_nudge(Grid G, StepPtrs S, int nudge) {
    const int i = blockIdx.x * BX + threadIdx.x, k = blockIdx.y * BY + threadIdx.y;
    if (i < 1 || i > G.nx - 2 || k < 1 || k > G.nz - 2) return;
    const size_t p = ix(G, i, k);
    const double rt = S.P.rate_th[k], rz = S.P.rate_z[k];
    if ((nudge & 1) && rt != 0.) S.fut[F_TH][p] -= rt * (S.fut[F_TH][p] - S.P.thb_init[k]);
    if ((nudge & 2) && rz != 0.) S.fut[F_ZETA][p] -= rz * (S.fut[F_ZETA][p]);
}

void launch_nudge(const Grid &G, const StepPtrs &S, int nudge, hipStream_t st) {
    hipLaunchKernelGGL(k_nudge, grid2d(G), dim3(BX, BY), 0, st, G, S, nudge);
}
void launch_nudge_qv(const Grid &G, const StepPtrs &S, double tau, hipStream_t st) {
    hipLaunchKernelGGL(k_nudge_qv, grid2d(G), dim3(BX, BY), 0, st, G, S, tau);
}
void launch_update_mean(const Grid &G, const StepPtrs &S, MeanMode mode, hipStream_t st) {
    hipLaunchKernelGGL(k_update_mean, dim3(G.nz - 2), dim3(256), 0, st, G, S, mode);
}

}  // namespace vvmd

// ------------------------------------------------ no-allocation entry point
//
// vvm_negative_value_noalloc runs the kernels of the handle's
// NegativeValueProcess operator (k_negval_sums, k_finalize, k_negval_scale)
// on a caller's device field.  Their scratch -- the two partial sums of each
// workgroup, then the correction ratio -- is the file-scope array below
// instead of a handle's buffers, so the call allocates nothing.  Every
// workgroup overwrites its own two partials and k_finalize reads only this
// call's workgroups and writes the ratio before k_negval_scale reads it, so
// nothing needs clearing between calls.  Calls that overlap on one GPU share
// the array and race.

namespace vvmd {
constexpr int kNoAllocMaxBlocks = 8192;  // 64x4-point workgroups: 2050x992 points at most
}  // namespace vvmd

static __device__ __align__(256) double scratch[2 * vvmd::kNoAllocMaxBlocks + 32];

namespace {
// Device address of `scratch` on each device, taken once with that device
// current (each GPU holds its own copy of the array at its own address).
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
double *g_scratch_ptr[kMaxDevices] = {};

int scratch_for_current_device(double **out) {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return VVM_ERR_HIP;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            fprintf(stderr, "vvm_negative_value_noalloc: hipGetSymbolAddress(scratch) on device %d: %s\n", dev,
                    hipGetErrorString(e));
            return VVM_ERR_HIP;
        }
        g_scratch_ptr[dev] = static_cast<double *>(p);
    }
    *out = g_scratch_ptr[dev];
    return VVM_OK;
}
}  // namespace

extern "C" int vvm_negative_value_noalloc(double *d_var, int nx, int nz, int pitch, void *stream) {
    using namespace vvmd;
    if (!d_var || nx < 3 || nz < 3 || pitch < nx) {
        fprintf(stderr, "vvm_negative_value_noalloc: bad arguments (var %p, nx %d, nz %d, pitch %d)\n",
                static_cast<void *>(d_var), nx, nz, pitch);
        return VVM_ERR_ARG;
    }
    Grid G{};
    G.nx = nx;
    G.nz = nz;
    G.pitch = pitch;
    const dim3 g = grid2d(G);
    const int nb = nblocks(g);
    if (nb > kNoAllocMaxBlocks) {
        fprintf(stderr,
                "vvm_negative_value_noalloc: a %d x %d field needs %d workgroups of %dx%d points; the "
                "no-allocation scratch holds %d (use vvm_dev_op_field for larger grids)\n",
                nx, nz, nb, BX, BY, kNoAllocMaxBlocks);
        return VVM_ERR_SIZE;
    }
    double *s = nullptr;
    if (const int rc = scratch_for_current_device(&s)) return rc;
    const RedSlot rs{s, kNoAllocMaxBlocks};
    double *ratio = s + 2 * kNoAllocMaxBlocks;
    hipStream_t st = static_cast<hipStream_t>(stream);
    hipLaunchKernelGGL(k_negval_sums, g, dim3(BX, BY), 0, st, G, d_var, rs);
    finalize<2>(rs, nb, ratio, RED_NEGVAL, 0, st);
    hipLaunchKernelGGL(k_negval_scale, g, dim3(BX, BY), 0, st, G, d_var, ratio);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        fprintf(stderr, "vvm_negative_value_noalloc: launch failed: %s\n", hipGetErrorString(e));
        return VVM_ERR_HIP;
    }
    return VVM_OK;
}
