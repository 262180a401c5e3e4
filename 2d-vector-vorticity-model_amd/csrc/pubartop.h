// pubartop.h -- pubarTop_pt as one workgroup's work, alone (k_pubartop) or
// beside the solve's first kernel (k_rows_fwd).
#pragma once

#include "vvm_internal.h"

namespace vvmd {

// PoissonSolver::pubarTop_pt (src/PoissonSolver.cpp:655-676): domain-mean
// vertical momentum flux and K_M shear at the top, AB2 for ubarTopp.  One
// workgroup, of any number of wavefronts.
__device__ inline void pubartop_block(const Grid &G, const StepPtrs &S, int step) {
#pragma clang fp contract(off)
    const int nx = G.nx, nz = G.nz;
    const double *u = S.u, *w = S.w, *K = S.RKM, *rhou = S.P.rhou, *rhow = S.P.rhow;
    double acc[3] = {0., 0., 0.};
    for (int i = 1 + threadIdx.x; i < nx - 1; i += blockDim.x) {
        acc[0] += 0.25 * (rhou[nz - 2] * u[ix(G, i, nz - 2)] + rhou[nz - 3] * u[ix(G, i, nz - 3)]) *
                  (w[ix(G, i, nz - 2)] + w[ix(G, i - 1, nz - 2)]);
        acc[1] += rhow[nz - 1] * 0.25 *
                  (K[ix(G, i, nz - 1)] + K[ix(G, i, nz - 2)] + K[ix(G, i - 1, nz - 1)] + K[ix(G, i - 1, nz - 2)]) *
                  (G.rdz * (u[ix(G, i, nz - 1)] - u[ix(G, i, nz - 2)]));
        acc[2] += rhow[nz - 2] * 0.25 *
                  (K[ix(G, i, nz - 2)] + K[ix(G, i, nz - 3)] + K[ix(G, i - 1, nz - 2)] + K[ix(G, i - 1, nz - 3)]) *
                  (G.rdx * (w[ix(G, i, nz - 2)] - w[ix(G, i - 1, nz - 2)]) +
                   G.rdz * (u[ix(G, i, nz - 2)] - u[ix(G, i, nz - 3)]));
    }
    block_sum<3>(acc);
    if (threadIdx.x == 0) {
        const double n = (double)(nx - 2.);
        const double down = acc[0] / n, kup = acc[1] / n, kdown = acc[2] / n;
        const double p1 = (-down) * G.rdz / rhou[nz - 2];
        const double p2 = (kup - kdown) * G.rdz / rhou[nz - 2];
        const int sn = (step + 1) % 2, so = step % 2;
        double *dub = S.s + S_DUBAR0;
        dub[sn] = -p1 + p2;
        if (step == 0) dub[0] = dub[1];
        S.s[S_UBARTOPP] = S.s[S_UBARTOP] + 1.5 * G.dt * dub[sn] - 0.5 * G.dt * dub[so];
    }
}

}  // namespace vvmd
