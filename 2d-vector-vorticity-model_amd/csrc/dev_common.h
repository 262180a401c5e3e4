// dev_common.h -- device layout and helpers shared by the VVM HIP kernels.
//
// Every 2-D model field lives x-contiguous on the device: element (i,k) of
// the reference's [i][k] array is at k*pitch + i, with i = 0..nx-1 and
// k = 0..nz-1 including the ghost cells.  Rows are padded to `pitch`
// elements (a multiple of 64) so every row starts 512-byte aligned.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace vvmd {

struct Grid {
    int nx, nz, pitch;
    double dx, dz, dt;
    double rdx, r2dx, rdz, r2dz, rdx2, rdz2;
    double GRAVITY, Cp, Cv, Rd, Lv, P0;
};

__host__ __device__ inline size_t ix(const Grid &G, int i, int k) { return size_t(k) * G.pitch + i; }

// Element (i,k) of a field, addressed as a row pointer plus a 32-bit byte
// offset.  Where k is the same for a whole wavefront (uniform), the row pointer
// stays in scalar registers and one vector register holds the offset for every
// field; with a 64-bit index per access half of a stencil kernel's vector
// instructions were address arithmetic.
__device__ inline double &at(double *a, const Grid &G, int i, int k) {
    return *reinterpret_cast<double *>(reinterpret_cast<char *>(a + size_t(k) * G.pitch) + unsigned(i) * 8u);
}
__device__ inline const double &at(const double *a, const Grid &G, int i, int k) {
    return *reinterpret_cast<const double *>(reinterpret_cast<const char *>(a + size_t(k) * G.pitch) +
                                             unsigned(i) * 8u);
}
// A value that is the same in every lane, as a scalar: threadIdx.y where
// blockDim.x is a wavefront.
__device__ inline int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// Stores v at interior point (i,k) and at every ghost cell that
// BoundaryProcess2D_center (src/Boundary.cpp:9-19) fills from it: the
// periodic column image for k in 1..nz-2, the zero-gradient row image at
// k = 1 / nz-2, and the corner that takes both.
__device__ inline void store_center(double *a, const Grid &G, int i, int k, double v) {
    at(a, G, i, k) = v;
    const bool west_img = (i == G.nx - 2), east_img = (i == 1);
    if (west_img) at(a, G, 0, k) = v;
    if (east_img) at(a, G, G.nx - 1, k) = v;
    if (k == 1) {
        at(a, G, i, 0) = v;
        if (west_img) at(a, G, 0, 0) = v;
        if (east_img) at(a, G, G.nx - 1, 0) = v;
    }
    if (k == G.nz - 2) {
        at(a, G, i, G.nz - 1) = v;
        if (west_img) at(a, G, 0, G.nz - 1) = v;
        if (east_img) at(a, G, G.nx - 1, G.nz - 1) = v;
    }
}

// Stores v at (i,k), k in 2..nz-2, plus its periodic column image, as
// BoundaryProcess2D_westdown (src/Boundary.cpp:21-31) does; rows 0, 1 and
// nz-1 are zero and are written by the caller.
__device__ inline void store_westdown(double *a, const Grid &G, int i, int k, double v) {
    at(a, G, i, k) = v;
    if (i == G.nx - 2) at(a, G, 0, k) = v;
    if (i == 1) at(a, G, G.nx - 1, k) = v;
}

// Notes the time in slot of clock, if there is one: the first workgroup's first
// thread as the kernel starts, or the last one's as it ends.
__device__ inline void note_time(long long *clock, int slot) {
    if (threadIdx.x == 0 && threadIdx.y == 0)
        __hip_atomic_store(clock + slot, (long long)wall_clock64(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
__device__ inline void note_start(long long *clock, int slot) {
    if (clock && blockIdx.x == 0 && blockIdx.y == 0) note_time(clock, slot);
}
__device__ inline void note_end(long long *clock, int slot) {
    if (clock && blockIdx.x == gridDim.x - 1 && blockIdx.y == gridDim.y - 1) note_time(clock, slot);
}

// A plane's value that the step does not touch again, past the caches if PAST.
template <bool PAST>
__device__ inline double load_once(const double &a) {
    if constexpr (PAST) return __builtin_nontemporal_load(&a);
    else return a;
}
template <bool PAST>
__device__ inline void store_once(double &a, double v) {
    if constexpr (PAST) __builtin_nontemporal_store(v, &a);
    else a = v;
}

// ---------------------------------------------------------------- sums

constexpr int kWave = 64;

// The value CTRL (a DPP control) brings from another lane, 0 where there is
// none or the row of 16 lanes is not in ROWS: a register move, where a shuffle
// is a round trip through LDS.
enum { DPP_ROW_SHR = 0x110, DPP_WAVE_SHR1 = 0x138, DPP_ROW_BCAST15 = 0x142, DPP_ROW_BCAST31 = 0x143 };
template <int CTRL, int ROWS = 0xf, typename T>
__device__ inline T dpp(T v) {
    static_assert(sizeof(T) == 4 || sizeof(T) == 8, "32 or 64 bits");
    int w[sizeof(T) / 4];
    __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
    for (int &x : w) x = __builtin_amdgcn_update_dpp(0, x, CTRL, ROWS, 0xf, true);
    __builtin_memcpy(&v, w, sizeof(T));
    return v;
}
// lane l's value, l uniform
template <typename T>
__device__ inline T from_lane(T v, int l) {
    int w[sizeof(T) / 4];
    __builtin_memcpy(w, &v, sizeof(T));
#pragma unroll
    for (int &x : w) x = __builtin_amdgcn_readlane(x, l);
    __builtin_memcpy(&v, w, sizeof(T));
    return v;
}

// Inclusive prefix sums over each row of 16 lanes, and over the wavefront.
template <typename T>
__device__ inline T row_scan(T v) {
    v += dpp<DPP_ROW_SHR + 1>(v);
    v += dpp<DPP_ROW_SHR + 2>(v);
    v += dpp<DPP_ROW_SHR + 4>(v);
    v += dpp<DPP_ROW_SHR + 8>(v);
    return v;
}
template <typename T>
__device__ inline T wave_scan(T v) {
    v = row_scan(v);
    v += dpp<DPP_ROW_BCAST15, 0xa>(v);
    v += dpp<DPP_ROW_BCAST31, 0xc>(v);
    return v;
}
template <typename T>
__device__ inline T wave_sum(T v) {
    return from_lane(wave_scan(v), kWave - 1);
}

// v[j] = sh[j][0] + .. + sh[j][n - 1], n <= W <= 16, in every lane: a row of
// lanes a value, four values at once.
template <int W, int NV, typename T>
__device__ inline void sum_rows(const T (&sh)[NV][W], int n, T (&v)[NV]) {
    const int lane = (threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z)) % kWave;
#pragma unroll
    for (int j0 = 0; j0 < NV; j0 += 4) {
        const int j = j0 + lane / 16;
        const T s = row_scan(j < NV && lane % 16 < n ? sh[min(j, NV - 1)][min(lane % 16, W - 1)] : T(0));
#pragma unroll
        for (int q = 0; q < 4; q++)
            if (j0 + q < NV) v[j0 + q] = from_lane(s, 16 * q + 15);
    }
}

// Block-wide sums of NV values; the totals are returned to every thread.
// blockDim must be a multiple of 64 and at most 1024, so that the wavefronts'
// sums of a value fit a row of lanes.  With shuffles and a loop over the wavefronts, two values over 1024
// threads took 2 us.
template <int NV, typename T>
__device__ inline void block_sum(T (&v)[NV]) {
    __shared__ T sh[NV][16];
    const int tid = threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z);
    const int nthr = blockDim.x * blockDim.y * blockDim.z;
    const int lane = tid % kWave, wid = tid / kWave, nw = nthr / kWave;
#pragma unroll
    for (int j = 0; j < NV; j++) v[j] = wave_sum(v[j]);
    if (lane == 0) {
#pragma unroll
        for (int j = 0; j < NV; j++) sh[j][wid] = v[j];
    }
    __syncthreads();
    sum_rows<16>(sh, nw, v);
    __syncthreads();
}

// Grid-wide FP64 sums are two launches: every block of the producing kernel
// writes its block sums with plain stores (block_partials), then one
// workgroup (k_finalize) adds them in block order and derives the scalars
// the next kernels read.  The kernel boundary orders the two; no fence or
// atomic is needed inside the producer.  (A last-block-done pattern needs an
// agent-scope release per block, which on a GPU with one L2 per XCD costs an
// L2 write-back each time.)  The order is fixed, so results are
// deterministic from run to run.
struct RedSlot {
    double *partial;  // [8][max_blocks]
    int max_blocks;
};

template <int NV>
__device__ inline void block_partials(double (&v)[NV], const RedSlot &rs, int bid) {
    const int tid = threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z);
    block_sum<NV>(v);
    if (tid == 0) {
#pragma unroll
        for (int j = 0; j < NV; j++) rs.partial[size_t(j) * rs.max_blocks + bid] = v[j];
    }
}
template <int NV>
__device__ inline void block_partials(double (&v)[NV], const RedSlot &rs) {
    block_partials<NV>(v, rs, blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z));
}

// Workgroups go round the 8 XCDs in turn, each with an L2 of its own.  Stencil
// kernels whose tiles share halos map them so that an XCD works one contiguous
// run of the n tiles (a band of rows): workgroup b of xcd_grid(n) takes tile
// xcd_tile(n), none if that is >= n.
constexpr int kXcds = 8;
__host__ __device__ inline int xcd_run(int n) { return (n + kXcds - 1) / kXcds; }
inline dim3 xcd_grid(int n) { return dim3(unsigned(kXcds * xcd_run(n))); }
__device__ inline int xcd_tile(int n) {
    const int b = blockIdx.x, run = xcd_run(n), t = (b % kXcds) * run + b / kXcds;
    return t;
}

// Scalars of the preconditioned CG (doubles in its scalar block).
// P_RZ / P_RZ2: r.z of odd / even CG iterations, P_ALPHA / P_ALPHA2 the
// step lengths of the single-reduction form (two slots each, so that the
// kernel forming the new value never overwrites the one its other
// workgroups still read).  Slot 1 is unused.
enum { P_RZ = 0, P_SPARE, P_ALPHA, P_ALPHA2, P_RNORM2, P_BNORM2, P_RNORM2_0, P_RZ2, NPSCAL = 8 };

// What k_finalize does with the totals.
enum RedMode {
    RED_STORE = 0,   // sc[dst+j] = tot[j] (and sc[dst2+j] when dst2 >= 0)
    RED_NEGVAL,      // NegativeValueProcess ratios of 3 fields into sc[dst+q]
    RED_RZ_INIT      // CG: sc[P_RZ] = rz
};

// NegativeValueProcess's ratio from the sums of the positives and negatives
// (MicroPhysics.cpp:129-131): no rescale when nothing is positive or the
// negatives outweigh the positives (marked by a ratio < 0).
__device__ inline double negval_ratio(double P, double N) {
    return (P == 0. || fabs(N) > P) ? -1. : 1. - fabs(N / P);
}

// The totals of nblk workgroups' partials, in every thread of a workgroup.
// They are added as by 256 threads, in a fixed order, whatever the workgroup's
// size: all callers agree bit for bit.
template <int NV>
__device__ inline void sum_partials(const RedSlot &rs, int nblk, double (&acc)[NV]) {
    __shared__ double sh[NV][4];
    const int tid = threadIdx.x + blockDim.x * threadIdx.y, nw = blockDim.x * blockDim.y / kWave;
    const int lane = tid % kWave, wid = tid / kWave;
    for (int vw = wid; vw < 4; vw += nw) {
#pragma unroll
        for (int j = 0; j < NV; j++) acc[j] = 0.;
#pragma unroll 4
        for (int b = vw * kWave + lane; b < nblk; b += 256) {
#pragma unroll
            for (int j = 0; j < NV; j++) acc[j] += rs.partial[size_t(j) * rs.max_blocks + b];
        }
#pragma unroll
        for (int j = 0; j < NV; j++) {
            const double t = wave_sum(acc[j]);
            if (lane == 0) sh[j][vw] = t;
        }
    }
    __syncthreads();
    sum_rows<4>(sh, 4, acc);
    __syncthreads();
}

namespace {
template <int NV>
__global__ void __launch_bounds__(256) k_finalize(RedSlot rs, int nblk, double *sc, int mode, int dst, int dst2,
                                                  double *hout) {
    double acc[NV];
    sum_partials<NV>(rs, nblk, acc);
    if (threadIdx.x != 0) return;
    switch (mode) {
        case RED_STORE:
            for (int j = 0; j < NV; j++) {
                sc[dst + j] = acc[j];
                if (dst2 >= 0) sc[dst2 + j] = acc[j];
                // host-mapped coherent memory: the host reads it after an
                // event, with no copy in the stream
                if (hout) __hip_atomic_store(hout + j, acc[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            }
            break;
        case RED_NEGVAL:
            for (int q = 0; q < NV / 2; q++) sc[dst + q] = negval_ratio(acc[2 * q], acc[2 * q + 1]);
            break;
        case RED_RZ_INIT:
            sc[P_RZ] = acc[0];
            break;
    }
}
}  // namespace

template <int NV>
inline void finalize(const RedSlot &rs, int nblk, double *sc, int mode, int dst, hipStream_t st, int dst2 = -1,
                     double *hout = nullptr) {
    hipLaunchKernelGGL(k_finalize<NV>, dim3(1), dim3(256), 0, st, rs, nblk, sc, mode, dst, dst2, hout);
}

// Sum of a grid's block partials (row 0 of rs, nblk of them) inside every
// block of the consuming kernel, in a fixed order, so that all blocks agree
// bit for bit; this saves a one-block k_finalize launch between producer
// and consumer when nblk is small.
__device__ inline double block_total(const RedSlot &rs, int nblk) {
    const int tid = threadIdx.x + blockDim.x * (threadIdx.y + blockDim.y * threadIdx.z);
    const int nthr = blockDim.x * blockDim.y * blockDim.z;
    double v[1] = {0.};
    for (int b = tid; b < nblk; b += nthr) v[0] += rs.partial[b];
    block_sum<1>(v);
    return v[0];
}

inline int nblocks(dim3 g) { return int(g.x * g.y * g.z); }

}  // namespace vvmd
