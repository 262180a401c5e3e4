// scale_forcing.h -- the second pass of NegativeValueProcess
// (MicroPhysics.cpp:129-137) and AddForcing (AddForcing.cpp:6-28) at one point,
// for k_scale_forcing and for k_kessler, which applies them as it reads.
#pragma once

#include "vvm_internal.h"

namespace vvmd {

// The three ratios: from the producing kernel's nblk partials in rs, added by
// every workgroup (256 threads), or (nblk = 0) the scalars k_finalize left.
__device__ inline void negval_ratios(const StepPtrs &S, const RedSlot &rs, int nblk, double (&ratios)[3]) {
    if (nblk > 0) {
        double acc[6];
        sum_partials<6>(rs, nblk, acc);
#pragma unroll
        for (int q = 0; q < 3; q++) ratios[q] = negval_ratio(acc[2 * q], acc[2 * q + 1]);
    } else {
#pragma unroll
        for (int q = 0; q < 3; q++) ratios[q] = S.s[S_NEG_RATIO + q];
    }
}

__device__ inline double rescaled(double v, double ratio) { return (ratio >= 0. && v > 0) ? v * ratio : v; }

// AddForcing's order (AddForcing.cpp:15-25): large-scale forcing, radiation
// heating [K/day], RADIATIONCOOLING, the random kick
__device__ inline double forced_th(const Grid &G, const StepPtrs &S, Forcing F, int i, int k, double th) {
#pragma clang fp contract(off)
    if (F.tropical) th += G.dt * S.P.Q1LS[k];
    if (S.rad) th += G.dt * at(S.rad, G, i, k) / 86400.;
    if (S.radcool) th += G.dt * (-2. / 86400.);
    if (F.random_kick) th += G.dt * at(S.forcing, G, i, k);
    return th;
}
__device__ inline double forced_qv(const Grid &G, const StepPtrs &S, Forcing F, int k, double qv) {
#pragma clang fp contract(off)
    if (F.tropical) qv += G.dt * S.P.Q2LS[k];
    return qv;
}

}  // namespace vvmd
