// micro.h -- the microphysics at one point: Kessler's processes, the second pass
// of NegativeValueProcess (MicroPhysics.cpp:129-137) and AddForcing
// (AddForcing.cpp:6-28), for kernels of their own (k_kessler, k_scale_forcing)
// and as further workgroups of the solve's (k_rows_fwd, k_columns).
#pragma once

#include "vvm_internal.h"

namespace vvmd {

// The three ratios: from the producing kernel's nblk partials in rs, added by
// every workgroup, or (nblk = 0) the scalars k_finalize left.
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

__device__ inline double rescaled(double v, double ratio) {
#pragma clang fp contract(off)
    return (ratio >= 0. && v > 0) ? v * ratio : v;
}

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

__device__ inline double maxs(double a, double b) { return (a < b) ? b : a; }
__device__ inline double mins(double a, double b) { return (b < a) ? b : a; }

// MicroPhysics::autoconversion, accretion, evaporation, condensation
// (MicroPhysics.cpp:29-51, 54-77, 80-114, 7-26).  Each is pointwise, so
// running the four in call order per point equals the reference's four
// sweeps.  Then the first pass of NegativeValueProcess on qvp, qcp, qrp
// (src/Iteration.cpp:309-311); k_finalize computes the three ratios.
// PROC selects the processes (KP_*); the timestep runs them all with the
// negative-value pass (KP_ALL).  One process alone (the reference's
// MicroPhysics statics) writes only the fields and the rate it changes.
// KP_PRE: the fields are read as thermo4 left them, and its negative-value
// rescale and AddForcing are applied on the way.  In the timestep that is one
// launch and one pass over four fields less, 9 us at 2048 x 256 between the
// advection and the solve: 20 steps there go 4948 -> 4806 us,
// 4096 x 256 8177 -> 7850.
// KP_PAST: the rates are written past the caches (past_caches).
enum { KP_AUTO = 1, KP_ACCR = 2, KP_EVAP = 4, KP_COND = 8, KP_NEG = 16, KP_ALL = 31, KP_PRE = 32, KP_PAST = 64 };

template <int PROC>
__device__ inline void kessler_point(const Grid &G, const StepPtrs &S, const Forcing &F, const double (&ratios)[3],
                                     int i, int k, double (&part)[6]) {
#pragma clang fp contract(off)
            const double dt = G.dt, pib = S.P.pib[k], rhou = S.P.rhou[k], pb = S.P.pb[k], pc = S.P.pcoef[k];
            double qc = at(S.fut[F_QC], G, i, k), qr = at(S.fut[F_QR], G, i, k), qv = at(S.fut[F_QV], G, i, k), th = at(S.fut[F_TH], G, i, k);
            if constexpr ((PROC & KP_PRE) != 0) {
                qv = forced_qv(G, S, F, k, rescaled(qv, ratios[0]));
                qc = rescaled(qc, ratios[1]);
                qr = rescaled(qr, ratios[2]);
                th = forced_th(G, S, F, i, k, th);
            }
            if constexpr ((PROC & KP_AUTO) != 0) {  // autoconversion
                const double qcplus = maxs(0., qc);
                double ar = 0.001 * (qcplus - 0.001);
                ar = maxs(0., ar);
                const double arcrdt = mins(ar * dt, qcplus);
                qc = qc - arcrdt;
                qr = qr + arcrdt;
                store_once<(PROC & KP_PAST) != 0>(at(S.autoc, G, i, k), arcrdt);
            }
            if constexpr ((PROC & KP_ACCR) != 0) {  // accretion
                const double qcplus = maxs(0., qc), qrplus = maxs(0., qr);
                // no rain, over most of a domain: the power is zero
                const double cr = 2.2 * qcplus * (qrplus == 0. ? 0. : pow(qrplus, 0.875));
                const double arcrdt = mins(cr * dt, qcplus);
                qc = qc - arcrdt;
                qr = qr + arcrdt;
                store_once<(PROC & KP_PAST) != 0>(at(S.accr, G, i, k), arcrdt);
            }
            if constexpr ((PROC & KP_EVAP) != 0) {  // rain evaporation
                const double qrplus = maxs(0., qr), qvplus = maxs(0., qv);
                double erdt = 0.;
                if (qrplus != 0.) {  // otherwise nothing evaporates: erdt = min(0, ..)
                    const double qvs = pc * exp(17.27 * (pib * th - 273.) / (pib * th - 36.));
                    const double deficit = maxs((1. - qvplus / qvs), 0.);
                    const double coef = 1.6 + 124.9 * pow((1E-3 * rhou * qrplus), 0.2046);
                    const double er = coef * deficit * (pow(1E-3 * rhou * qrplus, 0.525)) /
                                      ((5.4E5 + 2.55E6 / (1E-2 * pb * qvs)) * 1E-3 * rhou);
                    erdt = mins(qrplus, maxs(0., er * dt));
                }
                qr = qr - erdt;
                qv = qv + erdt;
                th = th - G.Lv * erdt / (G.Cp * pib);
                store_once<(PROC & KP_PAST) != 0>(at(S.evap, G, i, k), erdt);
            }
            if constexpr ((PROC & KP_COND) != 0) {  // saturation adjustment
                const double qvs = pc * exp(17.27 * (pib * th - 273.) / (pib * th - 36.));
                const double tm = th * pib - 36.;
                const double phi = qvs * (17.27 * 237. * G.Lv) / (G.Cp * (tm * tm));
                double C = (qv - qvs) / (1 + phi);
                if (fabs(C) > qc && C < 0) C = -qc;
                qv = qv - C;
                qc = qc + C;
                th = th + G.Lv / (G.Cp * pib) * C;
                store_once<(PROC & KP_PAST) != 0>(at(S.cond, G, i, k), C);
            }
            double q3[3] = {qv, qc, qr};
            if constexpr ((PROC & KP_NEG) != 0) {
#pragma unroll
                for (int q = 0; q < 3; q++) {
                    if (q3[q] >= 0.) part[2 * q] += q3[q];
                    else {
                        part[2 * q + 1] += q3[q];
                        q3[q] = 0.;
                    }
                }
            }
            constexpr bool wv = (PROC & (KP_EVAP | KP_COND | KP_NEG)) != 0;
            constexpr bool wc = (PROC & (KP_AUTO | KP_ACCR | KP_COND | KP_NEG)) != 0;
            constexpr bool wr = (PROC & (KP_AUTO | KP_ACCR | KP_EVAP | KP_NEG)) != 0;
            constexpr bool wt = (PROC & (KP_EVAP | KP_COND)) != 0;
            if (wv) at(S.fut[F_QV], G, i, k) = q3[0];
            if (wc) at(S.fut[F_QC], G, i, k) = q3[1];
            if (wr) at(S.fut[F_QR], G, i, k) = q3[2];
            if (wt) at(S.fut[F_TH], G, i, k) = th;
}

// Second pass of NegativeValueProcess for qv, qc, qr (MicroPhysics.cpp:
// 129-137), AddForcing (F.on), and the center halos of thp, qvp, qcp, qrp.
// halos == 0 is AddForcing alone (ratios < 0): interior thp and qvp only.
__device__ inline void scale_point(const Grid &G, const StepPtrs &S, const Forcing &F, const double (&ratios)[3],
                                   bool halos, int i, int k) {
#pragma clang fp contract(off)
#pragma unroll
    for (int q = 0; q < 3; q++) {
        const int f = F_QV + q;
        double v = rescaled(at(S.fut[f], G, i, k), ratios[q]);
        if (F.on && f == F_QV) v = forced_qv(G, S, F, k, v);
        if (halos) store_center(S.fut[f], G, i, k, v);
        else if (f == F_QV) at(S.fut[f], G, i, k) = v;
    }
    double th = at(S.fut[F_TH], G, i, k);
    if (F.on) th = forced_th(G, S, F, i, k, th);
    if (halos) store_center(S.fut[F_TH], G, i, k, th);
    else at(S.fut[F_TH], G, i, k) = th;
}

// The timestep's microphysics as workgroups of the solve's kernels, with
// 1-D blocks of whole wavefronts: each of the nblk workgroups walks tiles of 64
// columns and a row a wavefront.  First Kessler with KP_PRE (nv: thermo4's
// partials), leaving its own partials in rs; in a later launch the second pass.
struct Micro {
    Negval nv;
    Forcing F;
    RedSlot rs;
    int nblk = 0;
};
constexpr int kMicroBlocks = 512;
__device__ __host__ inline int micro_tiles(const Grid &G, int threads) {
    const int rows = threads / kWave;
    return ((G.nx - 2 + kWave - 1) / kWave) * ((G.nz - 2 + rows - 1) / rows);
}
template <typename P>
__device__ inline void micro_walk(const Grid &G, int block, int nblk, P point) {
    const int rows = blockDim.x / kWave, tx = (G.nx - 2 + kWave - 1) / kWave, nt = micro_tiles(G, blockDim.x);
    for (int t = block; t < nt; t += nblk) {
        const int i = 1 + (t % tx) * kWave + threadIdx.x % kWave;
        const int k = 1 + (t / tx) * rows + uniform(threadIdx.x / kWave);
        if (i <= G.nx - 2 && k <= G.nz - 2) point(i, k);
    }
}
__device__ inline void kessler_block(const Grid &G, const StepPtrs &S, const Micro &m, int block) {
    double part[6] = {0., 0., 0., 0., 0., 0.}, ratios[3];
    negval_ratios(S, m.nv.rs, m.nv.nblk, ratios);
    micro_walk(G, block, m.nblk,
               [&](int i, int k) { kessler_point<KP_ALL | KP_PRE>(G, S, m.F, ratios, i, k, part); });
    block_partials<6>(part, m.rs, block);
}
__device__ inline void scale_block(const Grid &G, const StepPtrs &S, const Negval &nv, int block, int nblk) {
    double ratios[3];
    negval_ratios(S, nv.rs, nv.nblk, ratios);
    micro_walk(G, block, nblk, [&](int i, int k) { scale_point(G, S, Forcing{}, ratios, true, i, k); });
}

}  // namespace vvmd
