// k_dynamics.hip -- advection, buoyancy, rain sedimentation, the negative
// value fixer, forcing and halos of one VVM timestep (phase A of
// vvm::Iteration::TimeMarching, src/Iteration.cpp:263-285), plus
// PoissonSolver::pubarTop_pt.
//
// FP64 throughout; no FMA contraction, so every expression rounds as the
// reference's does (the oracle and the compiled reference agree bit for bit
// on these operators; the GPU differs only where the device math library's
// pow/sqrt/exp do).
#pragma clang fp contract(off)

#include "pubartop.h"
#include "micro.h"
#include "vvm_internal.h"

namespace vvmd {

namespace {

constexpr int BX = 64, BY = 4;

__device__ inline double plus_(double v) { return 0.5 * (v + fabs(v)); }
__device__ inline double minu_(double v) { return 0.5 * (v - fabs(v)); }

// Third-order upwind-biased correction of one face flux, Advection.cpp:40-50
// (rho0/v0 at the face, rhom/vm one face upstream, rhop/vp one downstream;
// fm2..fp1 the four cell values around the face).
__device__ inline double upwind3(double rho0, double v0, double rhom, double vm, double rhop, double vp, double fm2,
                                 double fm1, double f0, double fp1) {
    const double p0 = plus_(v0), pm = plus_(vm), m0 = minu_(v0), mp = minu_(vp);
    return -1. / 3. *
           (rho0 * p0 * (f0 - fm1) - sqrt(rho0 * p0 * rhom * pm) * (fm1 - fm2) - rho0 * m0 * (f0 - fm1) -
            sqrt(fabs(rho0 * m0 * rhop * mp)) * (fp1 - f0));
}

__device__ inline bool corr_window(const Grid &G, int i, int k) {
    return i >= 2 && i <= G.nx - 3 && k >= 2 && k <= G.nz - 3;
}

// Scalar x-face flux at (i,k) (between i-1 and i), Advection.cpp:36,40-44.
__device__ inline double sflux_x(const Grid &G, const double *__restrict__ f, const double *__restrict__ u,
                                 const double *__restrict__ rhou, int i, int k) {
    const double r = rhou[k], ui = at(u, G, i, k);
    const double f0 = at(f, G, i, k), fm1 = at(f, G, i - 1, k);
    double fl = r * ui * (f0 + fm1);
    if (corr_window(G, i, k))
        fl += upwind3(r, ui, r, at(u, G, i - 1, k), r, at(u, G, i + 1, k), at(f, G, i - 2, k), fm1, f0,
                      at(f, G, i + 1, k));
    return fl;
}

// Scalar z-face flux at (i,k) (between k-1 and k), Advection.cpp:37,46-50.
__device__ inline double sflux_z(const Grid &G, const double *__restrict__ f, const double *__restrict__ w,
                                 const double *__restrict__ rhow, int i, int k) {
    const double r = rhow[k], wk = at(w, G, i, k);
    const double f0 = at(f, G, i, k), fm1 = at(f, G, i, k - 1);
    double fl = r * wk * (f0 + fm1);
    if (corr_window(G, i, k))
        fl += upwind3(r, wk, rhow[k - 1], at(w, G, i, k - 1), rhow[k + 1], at(w, G, i, k + 1), at(f, G, i, k - 2),
                      fm1, f0, at(f, G, i, k + 1));
    return fl;
}

// Corner velocities of Advection_zeta, Advection.cpp:90-91.
__device__ inline double Uw(const Grid &G, const double *u, const double *rhou, int i, int k) {
    return 0.25 * (rhou[k] * (at(u, G, i + 1, k) + at(u, G, i, k)) +
                   rhou[k - 1] * (at(u, G, i + 1, k - 1) + at(u, G, i, k - 1)));
}
__device__ inline double Wu(const Grid &G, const double *w, const double *rhow, int i, int k) {
    return 0.25 * (rhow[k + 1] * (at(w, G, i, k + 1) + at(w, G, i - 1, k + 1)) +
                   rhow[k] * (at(w, G, i, k) + at(w, G, i - 1, k)));
}

// Vorticity fluxes, Advection.cpp:107-118 (the density already sits in U_w/W_u).
// The correction's values are read everywhere, at clamped indices, and dropped
// outside its window: loads in a branch are waited for before the next ones.
__device__ inline double zflux_x(const Grid &G, const double *z, const double *u, const double *rhou, int i, int k) {
    const double U = Uw(G, u, rhou, i, k), Um = Uw(G, u, rhou, i - 1, k);
    const double Up = Uw(G, u, rhou, min(i + 1, G.nx - 2), k);
    const double z0 = at(z, G, i, k), z1 = at(z, G, i + 1, k), zm = at(z, G, i - 1, k);
    const double z2 = at(z, G, min(i + 2, G.nx - 1), k);
    const double fl = U * (z1 + z0);
    const double Pu = plus_(U), Pum = plus_(Um), Mu = minu_(U), Mup = minu_(Up);
    const double cor = fl + -1. / 3. * (Pu * (z1 - z0) - sqrt(Pu * Pum) * (z0 - zm) - Mu * (z1 - z0) -
                                        sqrt(fabs(Mu * Mup)) * (z2 - z1));
    return corr_window(G, i, k) ? cor : fl;
}
__device__ inline double zflux_z(const Grid &G, const double *z, const double *w, const double *rhow, int i, int k) {
    const double W = Wu(G, w, rhow, i, k), Wm = Wu(G, w, rhow, i, k - 1);
    const double Wp = Wu(G, w, rhow, i, min(k + 1, G.nz - 2));
    const double z0 = at(z, G, i, k), z1 = at(z, G, i, k + 1), zm = at(z, G, i, k - 1);
    const double z2 = at(z, G, i, min(k + 2, G.nz - 1));
    const double fl = W * (z1 + z0);
    const double Pw = plus_(W), Pwm = plus_(Wm), Mw = minu_(W), Mwp = minu_(Wp);
    const double cor = fl + -1. / 3. * (Pw * (z1 - z0) - sqrt(Pw * Pwm) * (z0 - zm) - Mw * (z1 - z0) -
                                        sqrt(fabs(Mw * Mwp)) * (z2 - z1));
    return corr_window(G, i, k) ? cor : fl;
}

__device__ inline double thv(const Grid &G, const double *th, const double *qv, int i, int k) {
    return at(th, G, i, k) * (1 + 0.608 * at(qv, G, i, k));
}

// AB2 update of one history slot: writes d to slot sn (and to slot 0 on the
// reference's step-0 start, Advection.cpp:70) and returns the old slot.
template <bool PAST = false>
__device__ inline double ab2_hist(double *const (&h)[2], const Grid &G, int i, int k, int step, double d) {
    // the slot pointers are picked by selects, not by a run-time index into
    // the kernel-argument array (which would read them through generic
    // memory accesses)
    const bool odd = (step & 1) != 0;
    double *const hn = odd ? h[0] : h[1], *const ho = odd ? h[1] : h[0];
    store_once<PAST>(at(hn, G, i, k), d);
    if (step == 0) at(h[0], G, i, k) = d;
    return load_once<PAST>(at(ho, G, i, k));
}

// ------------------------------------------------------------------ zeta

// Iteration::pzeta_pt: Advection_zeta (Advection.cpp:84-149) + Bouyancy
// (Buoyancy.cpp:11-58) + BoundaryProcess2D_westdown(zetap).  As in
// k_thermo4, each vorticity flux is formed once per face: every thread forms
// the flux on its own east and upper faces, the first two waves the faces on
// the tile's west and lower edges, and after a barrier each point takes the
// differences.
// The tiles start at the first point that the advection changes (k = 2).
constexpr int PZX = 64, PZY = 8;
__host__ __device__ inline int pz_tiles_x(const Grid &G) { return (G.nx - 2 + PZX - 1) / PZX; }
__host__ __device__ inline int pz_tiles_z(const Grid &G) { return (G.nz - 3 + PZY - 1) / PZY; }

// PARTS: PZ_ADV Advection_zeta, PZ_BUOY Bouyancy; both (the timestep) also
// apply BoundaryProcess2D_westdown.  Alone each writes what the reference
// function writes: the interior points k = 2..nz-2 (zetap = ... for the
// advection, zetap += ... for the buoyancy) and its AB2 history.
enum { PZ_ADV = 1, PZ_BUOY = 2, PZ_BOTH = 3 };

struct PzLds {
    double Fx[PZY][PZX + 1];  // slot c: x-flux east of column i0 + c - 1
    double Fz[PZY + 1][PZX];  // slot r: z-flux above row k0 + r - 1
};
template <int PARTS, bool PAST>
__device__ inline void pzeta_tile(const Grid &G, const StepPtrs &S, int step, int tile, PzLds &lds) {
    auto &Fx = lds.Fx;
    auto &Fz = lds.Fz;
    const int tx = threadIdx.x, ty = uniform(threadIdx.y);  // PZX = T4X = 64: one row a wavefront
    const int tiles_x = pz_tiles_x(G);
    const int i0 = 1 + (tile % tiles_x) * PZX, k0 = 2 + (tile / tiles_x) * PZY;
    const int i = i0 + tx, k = k0 + ty;
    const int nx = G.nx, nz = G.nz;
    const double *z = S.now[F_ZETA], *u = S.u, *w = S.w, *rhou = S.P.rhou, *rhow = S.P.rhow;
    if constexpr ((PARTS & PZ_ADV) != 0) {
        if (k <= nz - 2 && i <= nx - 2) {
            Fx[ty][tx + 1] = zflux_x(G, z, u, rhou, i, k);
            Fz[ty + 1][tx] = zflux_z(G, z, w, rhow, i, k);
        }
        if (ty == 0 && tx < PZY) {  // west edge: the face east of column i0 - 1
            const int kr = k0 + tx;
            // east of column 0: the periodic image of nx-2
            // (BoundaryProcess2D_center on flux_u)
            if (kr <= nz - 2) Fx[tx][0] = zflux_x(G, z, u, rhou, (i0 == 1) ? nx - 2 : i0 - 1, kr);
        } else if (ty == 1) {  // lower edge: the face above row k0 - 1
            if (i <= nx - 2) Fz[0][tx] = zflux_z(G, z, w, rhow, i, k0 - 1);
        }
        __syncthreads();
    }
    double *zp = S.fut[F_ZETA];
    if (PARTS == PZ_BOTH && (ty == 0 || ty == 1) && i <= nx - 2) {
        // the zero rows 0, 1 (first tiles) and nz-1 (last tiles), ghosts included
        const bool first = k0 == 2, last = k0 + PZY > nz - 2;
        const int kz = (ty == 0) ? 0 : 1;
        auto clear = [&](int kc) {
            at(zp, G, i, kc) = 0.;
            if (i == 1) at(zp, G, 0, kc) = 0.;
            if (i == nx - 2) at(zp, G, nx - 1, kc) = 0.;
        };
        if (first) clear(kz);
        if (last && ty == 0) clear(nz - 1);
    }
    if (i > nx - 2 || k > nz - 2) return;
    double zeta_new;
    if constexpr ((PARTS & PZ_ADV) != 0) {
        const double fu0 = Fx[ty][tx + 1], fum = Fx[ty][tx];
        const double fw0 = Fz[ty + 1][tx], fwm = Fz[ty][tx];
        const double px = (fu0 - fum) * G.r2dx / rhow[k];
        const double pz = (fw0 - fwm) * G.r2dz / rhow[k];
        const double dadv = -px - pz;
        const double dold = ab2_hist<PAST>(S.hist[H_ZETA_ADV], G, i, k, step, dadv);
        zeta_new = at(z, G, i, k) + 1.5 * G.dt * dadv - 0.5 * G.dt * dold;
        if constexpr (PARTS == PZ_ADV) {
            at(zp, G, i, k) = zeta_new;
            return;
        }
    } else {
        zeta_new = at(zp, G, i, k);
    }

    const double *th = S.now[F_TH], *qv = S.now[F_QV], *qc = S.now[F_QC], *qr = S.now[F_QR], *thvb = S.P.thvb;
    const double gth = G.GRAVITY / rhow[k] * 0.5 *
                       ((thv(G, th, qv, i, k) - thv(G, th, qv, i - 1, k)) / thvb[k] +
                        (thv(G, th, qv, i, k - 1) - thv(G, th, qv, i - 1, k - 1)) / thvb[k - 1]) *
                       G.rdx;
    const double gqc = G.GRAVITY / rhow[k] *
                       (0.5 * (at(qc, G, i, k) + at(qc, G, i, k - 1)) - 0.5 * (at(qc, G, i - 1, k) + at(qc, G, i - 1, k - 1))) *
                       G.rdx;
    const double gqr = G.GRAVITY / rhow[k] *
                       (0.5 * (at(qr, G, i, k) + at(qr, G, i, k - 1)) - 0.5 * (at(qr, G, i - 1, k) + at(qr, G, i - 1, k - 1))) *
                       G.rdx;
    double db = gth;
    db += -gqc - gqr;
    const double bold = ab2_hist<PAST>(S.hist[H_TH_BUOY], G, i, k, step, db);
    zeta_new += (1.5 * G.dt * db) - (0.5 * G.dt * bold);
    if constexpr (PARTS == PZ_BOTH) store_westdown(zp, G, i, k, zeta_new);
    else at(zp, G, i, k) = zeta_new;
}
template <int PARTS, bool PAST = false>
__global__ void __launch_bounds__(PZX *PZY) k_pzeta(Grid G, StepPtrs S, int step) {
    note_start(S.clock, CLK_ADVECT);
    __shared__ PzLds lds;
    const int nt = pz_tiles_x(G) * pz_tiles_z(G), tile = xcd_tile(nt);
    if (tile < nt) pzeta_tile<PARTS, PAST>(G, S, step, tile, lds);
}

// ----------------------------------------------------------- scalars

// Advection_thermo (Advection.cpp:25-81) for one field at interior (i,k).
__device__ inline double thermo_tend(const Grid &G, const double *f, const double *u, const double *w,
                                     const double *rhou, const double *rhow, int i, int k) {
    const double fu1 = sflux_x(G, f, u, rhou, (i + 1 == G.nx - 1) ? 1 : i + 1, k);
    const double fu0 = sflux_x(G, f, u, rhou, i, k);
    const double fw1 = (k + 1 == G.nz - 1) ? 0. : sflux_z(G, f, w, rhow, i, k + 1);
    const double fw0 = sflux_z(G, f, w, rhow, i, k);
    const double px = (fu1 - fu0) * G.r2dx / rhou[k];
    const double pz = (fw1 - fw0) * G.r2dz / rhou[k];
    return -px - pz;
}

// The parts of a scalar face flux that depend only on the face (density and
// velocity), formed once and applied to every field advected across it.
// flux(f) rounds exactly as sflux_x / sflux_z do: the same products in the
// same order (upwind3's rho0 p0 (f0 - fm1) is (rho0 p0) (f0 - fm1), and so on).
template <bool X>  // an x face (between i-1 and i) or a z face (between k-1 and k)
struct FaceFlux {
    double rv;          // r v of the centred term
    double a, b, c, d;  // rho0 p0, sqrt(rho0 p0 rhom pm), rho0 m0, sqrt(|rho0 m0 rhop mp|)
    bool corr;          // inside the third-order correction window
    __device__ double flux(const Grid &G, const double *__restrict__ f, int i, int k) const {
        const double f0 = at(f, G, i, k), fm1 = X ? at(f, G, i - 1, k) : at(f, G, i, k - 1);
        const double fm2 = X ? at(f, G, max(i - 2, 0), k) : at(f, G, i, max(k - 2, 0));
        const double fp1 = X ? at(f, G, i + 1, k) : at(f, G, i, k + 1);
        const double fl = rv * (f0 + fm1);
        const double cor = fl + -1. / 3. * (a * (f0 - fm1) - b * (fm1 - fm2) - c * (f0 - fm1) - d * (fp1 - f0));
        return corr ? cor : fl;
    }
};
template <bool X>
__device__ inline FaceFlux<X> face_coeffs(double rho0, double v0, double rhom, double vm, double rhop, double vp,
                                          bool corr) {
    FaceFlux<X> F;
    const double p0 = plus_(v0), pm = plus_(vm), m0 = minu_(v0), mp = minu_(vp);
    F.rv = rho0 * v0;
    F.corr = corr;
    F.a = rho0 * p0;
    F.b = sqrt(F.a * rhom * pm);
    F.c = rho0 * m0;
    F.d = sqrt(fabs(F.c * rhop * mp));
    return F;
}
// x face between i-1 and i / z face between k-1 and k, as sflux_x / sflux_z,
// of an interior point; the correction's values are read everywhere and dropped
// outside its window (as in zflux_x)
__device__ inline FaceFlux<true> face_x(const Grid &G, const double *u, const double *rhou, int i, int k) {
    const double r = rhou[k];
    return face_coeffs<true>(r, at(u, G, i, k), r, at(u, G, i - 1, k), r, at(u, G, i + 1, k), corr_window(G, i, k));
}
__device__ inline FaceFlux<false> face_z(const Grid &G, const double *w, const double *rhow, int i, int k) {
    return face_coeffs<false>(rhow[k], at(w, G, i, k), rhow[k - 1], at(w, G, i, k - 1), rhow[k + 1],
                              at(w, G, i, k + 1), corr_window(G, i, k));
}

// Rain sedimentation flux of Advection_qrVT (Advection.cpp:165-166) at (i,k).
__device__ inline double vt_flux(const Grid &G, const double *qr, const double *rhow, const double *vtfac, int i,
                                 int k) {
    const double s = at(qr, G, i, k) + at(qr, G, i, k - 1);
    if (s == 0.) return s;  // no rain, over most of a domain: VT is zero, and pow is a third of the kernel
    const double VT = 1E-2 * (3634 * pow(1E-3 * rhow[k] * 0.5 * s, 0.1346) * vtfac[k]);
    return rhow[k] * VT * s;
}

// pth_pt, pqv_pt, pqc_pt, pqr_pt (src/Iteration.cpp:36-40, 90-124): the four
// scalar advections sharing u and w, rain sedimentation on qr, surface
// precipitation, and the first pass of NegativeValueProcess (zero the
// negatives, sum positives and negatives) for qv, qc, qr.  k_finalize turns
// the sums into rescale ratios.
//
// Each face flux is formed once, as the reference forms its flux arrays:
// a workgroup covers T4X x T4Y points; first every thread forms the x-face
// flux on its west face and the z-face fluxes (four fields and the rain
// fall) on its lower face, and a few waves form the faces on the tile's east
// and top edges; after a barrier each point takes the differences.  (Forming
// both faces of every point would evaluate each flux, with its square roots
// and powers, twice.)
// Small grids are one round of latencies: with the correction's loads ahead of
// its branch and the edge faces over six waves 13.6 -> 11.5 us at 128 x 64 and,
// with less serial work, 28.0 -> 25.9 at 2048 x 256.
// The tiles start at the first interior point: 2048 x 256 are 1024 of them, one
// round at four workgroups a CU.  (From the ghost cells on they were 1089, and
// the last 65 took a round of their own.)
constexpr int T4X = 64, T4Y = 8;
__host__ __device__ inline int t4_tiles_x(const Grid &G) { return (G.nx - 2 + T4X - 1) / T4X; }
__host__ __device__ inline int t4_tiles_z(const Grid &G) { return (G.nz - 2 + T4Y - 1) / T4Y; }

struct T4Lds {
    double Fx[4][T4Y][T4X + 1];  // x-face flux at faces i0 .. i0+T4X (west faces)
    double Fz[5][T4Y + 1][T4X];  // z-face flux (4 fields, rain fall) at faces k0 .. k0+T4Y
};
template <bool PAST>
__device__ inline void thermo4_tile(const Grid &G, const StepPtrs &S, int step, const RedSlot &rs, int tile, T4Lds &lds) {
    auto &Fx = lds.Fx;
    auto &Fz = lds.Fz;
    const int tx = threadIdx.x, ty = uniform(threadIdx.y);  // PZX = T4X = 64: one row a wavefront
    const int tiles_x = t4_tiles_x(G);
    const int i0 = 1 + (tile % tiles_x) * T4X, k0 = 1 + (tile / tiles_x) * T4Y;
    const int i = i0 + tx, k = k0 + ty;
    const int nx = G.nx, nz = G.nz;
    const double *u = S.u, *w = S.w, *rhou = S.P.rhou, *rhow = S.P.rhow;
    const double *fl[4] = {S.now[F_TH], S.now[F_QV], S.now[F_QC], S.now[F_QR]};
    const bool row_in = (k >= 1 && k <= nz - 2), inside = row_in && i >= 1 && i <= nx - 2;
    // the ghost column nx-1 holds the face east of column nx-2: the
    // periodic image of face 1
    // the density-velocity part of each face is formed once for all four
    // fields (sflux_x / sflux_z per field would repeat its square roots)
    if (row_in && i >= 1 && i <= nx - 1) {
        const int ii = (i == nx - 1) ? 1 : i;
        const FaceFlux<true> F = face_x(G, u, rhou, ii, k);
#pragma unroll
        for (int q = 0; q < 4; q++) Fx[q][ty][tx] = F.flux(G, fl[q], ii, k);
    }
    if (inside) {
        const FaceFlux<false> F = face_z(G, w, rhow, i, k);
#pragma unroll
        for (int q = 0; q < 4; q++) Fz[q][ty][tx] = F.flux(G, fl[q], i, k);
        Fz[4][ty][tx] = vt_flux(G, fl[3], rhow, S.P.vtfac, i, k);
    }
    // edge faces: waves 0-3 the top faces, one field each, wave 4 the top
    // rain-fall faces, wave 5 the east faces, eight lanes (rows) a field
    {
        const int kt = k0 + T4Y, ie = i0 + T4X;
        if (ty < 4) {
            if (i <= nx - 2 && kt <= nz - 2)
                Fz[ty][T4Y][tx] = face_z(G, w, rhow, i, kt).flux(G, S.now[F_TH + ty], i, kt);
        } else if (ty == 4) {
            if (i <= nx - 2 && kt <= nz - 2) Fz[4][T4Y][tx] = vt_flux(G, fl[3], rhow, S.P.vtfac, i, kt);
        } else if (ty == 5 && tx < 4 * T4Y) {
            const int q = tx / T4Y, r = tx % T4Y, kr = k0 + r;
            // the face east of column nx-2 is the periodic image of face 1
            if (ie - 1 <= nx - 2 && kr <= nz - 2) {
                const int ii = (ie == nx - 1) ? 1 : ie;
                const double *f = q < 2 ? (q == 0 ? fl[0] : fl[1]) : (q == 2 ? fl[2] : fl[3]);
                Fx[q][r][T4X] = face_x(G, u, rhou, ii, kr).flux(G, f, ii, kr);
            }
        }
    }
    __syncthreads();
    double part[6] = {0., 0., 0., 0., 0., 0.};
    if (inside) {
        const int hid[4] = {H_TH_ADV, H_QV_ADV, H_QC_ADV, H_QR_ADV};
        const bool top = (k + 1 == nz - 1);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            // Advection_thermo's tendency (Advection.cpp:55-81)
            const double fu1 = Fx[q][ty][tx + 1], fu0 = Fx[q][ty][tx];
            const double fw1 = top ? 0. : Fz[q][ty + 1][tx];
            const double fw0 = Fz[q][ty][tx];
            const double px = (fu1 - fu0) * G.r2dx / rhou[k];
            const double pz = (fw1 - fw0) * G.r2dz / rhou[k];
            const double d = -px - pz;
            const double dold = ab2_hist<PAST>(S.hist[hid[q]], G, i, k, step, d);
            double v = at(fl[q], G, i, k) + 1.5 * G.dt * d - 0.5 * G.dt * dold;
            if (q == 0) {
                at(S.fut[F_TH], G, i, k) = v;
                continue;
            }
            if (q == 3) {
                const double f1 = top ? 0. : Fz[4][ty + 1][tx];
                const double f0 = Fz[4][ty][tx];
                const double dvt = (f1 - f0) * G.r2dz / rhou[k];
                const double vold = ab2_hist<PAST>(S.hist[H_QR_VT], G, i, k, step, dvt);
                v += 1.5 * G.dt * dvt - 0.5 * G.dt * vold;
            }
            if (v >= 0.) part[2 * (q - 1)] += v;
            else {
                part[2 * (q - 1) + 1] += v;
                v = 0.;
            }
            at(S.fut[F_QV + q - 1], G, i, k) = v;
        }
        if (k == 1) {
            // surface precipitation, src/Iteration.cpp:114-119 (now-qr, last w)
            const double r1 = rhou[1];
            const double q1 = at(S.now[F_QR], G, i, 1);
            const double VT = 1E-2 * (3634 * pow(1E-3 * r1 * q1, 0.1346) * S.s[S_PRECIP_FAC]);
            const double rain = -r1 * (0.5 * (at(w, G, i, 2) + 0.) - VT) * q1;
            S.precip[i] = (rain < 0) ? 0. : rain;
        }
    }
    block_partials<6>(part, rs, tile);
}
// Four workgroups a CU (the LDS allows four), so that 1024 of them cover
// 2048 x 256 in one round: eight waves a SIMD, at most 64 VGPRs.
template <bool PAST>
__global__ void __launch_bounds__(T4X *T4Y) __attribute__((amdgpu_waves_per_eu(8)))
k_thermo4(Grid G, StepPtrs S, int step, RedSlot rs) {
    __shared__ T4Lds lds;
    const int nt = t4_tiles_x(G) * t4_tiles_z(G), tile = xcd_tile(nt);
    if (tile < nt) thermo4_tile<PAST>(G, S, step, rs, tile, lds);
}

// Both in one launch, a tile of each in turn: neither reads what the other
// writes, and the second of a pair finds the winds and scalars in its XCD's L2.
static_assert(T4X == PZX && T4Y == PZY, "one block shape");
__global__ void __launch_bounds__(T4X *T4Y) __attribute__((amdgpu_waves_per_eu(8)))
k_advect(Grid G, StepPtrs S, int step, RedSlot rs) {
    __shared__ union Lds {
        T4Lds t4;
        PzLds pz;
    } lds;
    note_start(S.clock, CLK_ADVECT);
    const int nt = t4_tiles_x(G) * t4_tiles_z(G), slot = xcd_tile(2 * nt), tile = slot / 2;
    if (slot >= 2 * nt) return;
    if (slot % 2 == 0) thermo4_tile<false>(G, S, step, rs, tile, lds.t4);
    else if (tile < pz_tiles_x(G) * pz_tiles_z(G)) pzeta_tile<PZ_BOTH, false>(G, S, step, tile, lds.pz);
}

__global__ void __launch_bounds__(BX *BY) k_scale_forcing(Grid G, StepPtrs S, Negval nv, Forcing F, int halos) {
    const int i = 1 + blockIdx.x * BX + threadIdx.x, k = 1 + blockIdx.y * BY + uniform(threadIdx.y);
    double ratios[3];
    negval_ratios(S, nv.rs, nv.nblk, ratios);
    if (i <= G.nx - 2 && k <= G.nz - 2) scale_point(G, S, F, ratios, halos != 0, i, k);
    note_end(S.clock, CLK_MICRO_END);
}

// Halo value of BoundaryProcess2D_center at a perimeter cell.
__device__ inline size_t center_src(const Grid &G, int i, int k) {
    const int is = (i == 0) ? G.nx - 2 : (i == G.nx - 1) ? 1 : i;
    const int ks = (k == 0) ? 1 : (k == G.nz - 1) ? G.nz - 2 : k;
    return ix(G, is, ks);
}

// BoundaryProcess2D_center / _westdown on the perimeter of a field.
__device__ inline void bc_center_cell(double *a, const Grid &G, int i, int k) {
    if (i == 0 || i == G.nx - 1 || k == 0 || k == G.nz - 1) at(a, G, i, k) = a[center_src(G, i, k)];
}
__device__ inline void bc_westdown_cell(double *a, const Grid &G, int i, int k) {
    if (k == 0 || k == 1 || k == G.nz - 1) at(a, G, i, k) = 0.;
    else if (i == 0) at(a, G, i, k) = at(a, G, G.nx - 2, k);
    else if (i == G.nx - 1) at(a, G, i, k) = at(a, G, 1, k);
}

__global__ void __launch_bounds__(BX *BY) k_bc_uw(Grid G, StepPtrs S) {
    const int i = blockIdx.x * BX + threadIdx.x, k = blockIdx.y * BY + uniform(threadIdx.y);
    if (i >= G.nx || k >= G.nz) return;
    bc_center_cell(S.u, G, i, k);
    bc_westdown_cell(S.w, G, i, k);
}

// BoundaryProcess2D_all (src/Boundary.cpp:33-52), Kessler build.
__global__ void __launch_bounds__(BX *BY) k_bc_all(Grid G, StepPtrs S) {
    const int i = blockIdx.x * BX + threadIdx.x, k = blockIdx.y * BY + uniform(threadIdx.y);
    if (i >= G.nx || k >= G.nz) return;
    bc_westdown_cell(S.fut[F_ZETA], G, i, k);
    bc_center_cell(S.fut[F_TH], G, i, k);
    bc_westdown_cell(S.w, G, i, k);
    bc_center_cell(S.u, G, i, k);
    bc_center_cell(S.fut[F_QV], G, i, k);
    bc_center_cell(S.fut[F_QC], G, i, k);
    bc_center_cell(S.fut[F_QR], G, i, k);
}

// ------------------------------------------------ single operators alone
// (the statics of class vvm one at a time; the timestep uses the fused
// kernels above).  Each writes exactly what its reference function writes.

// Advection_thermo (Advection.cpp:25-81) of field q (F_TH..F_QR): the
// interior of its p-field and its AB2 history.
__global__ void __launch_bounds__(BX *BY) k_adv_scalar(Grid G, StepPtrs S, int step, int q) {
    const int i = blockIdx.x * BX + threadIdx.x, k = blockIdx.y * BY + uniform(threadIdx.y);
    if (i < 1 || i > G.nx - 2 || k < 1 || k > G.nz - 2) return;
    const int hid[NPROG] = {H_ZETA_ADV, H_TH_ADV, H_QV_ADV, H_QC_ADV, H_QR_ADV};
    const double *f = S.now[q];
    const double d = thermo_tend(G, f, S.u, S.w, S.P.rhou, S.P.rhow, i, k);
    const double dold = ab2_hist(S.hist[hid[q]], G, i, k, step, d);
    at(S.fut[q], G, i, k) = at(f, G, i, k) + 1.5 * G.dt * d - 0.5 * G.dt * dold;
}

// Advection_qrVT (Advection.cpp:153-192): the rain fall added to the
// interior of qrp, and its AB2 history.
__global__ void __launch_bounds__(BX *BY) k_qrvt(Grid G, StepPtrs S, int step) {
    const int i = blockIdx.x * BX + threadIdx.x, k = blockIdx.y * BY + uniform(threadIdx.y);
    if (i < 1 || i > G.nx - 2 || k < 1 || k > G.nz - 2) return;
    const double *qr = S.now[F_QR], *rhow = S.P.rhow;
    const double f1 = (k + 1 == G.nz - 1) ? 0. : vt_flux(G, qr, rhow, S.P.vtfac, i, k + 1);
    const double f0 = vt_flux(G, qr, rhow, S.P.vtfac, i, k);
    const double dvt = (f1 - f0) * G.r2dz / S.P.rhou[k];
    const double vold = ab2_hist(S.hist[H_QR_VT], G, i, k, step, dvt);
    at(S.fut[F_QR], G, i, k) += 1.5 * G.dt * dvt - 0.5 * G.dt * vold;
}

// Surface precipitation of pqr_pt (src/Iteration.cpp:114-119).
__global__ void k_precip(Grid G, StepPtrs S) {
    const int i = 1 + blockIdx.x * blockDim.x + threadIdx.x;
    if (i > G.nx - 2) return;
    const double r1 = S.P.rhou[1], q1 = at(S.now[F_QR], G, i, 1);
    const double VT = 1E-2 * (3634 * pow(1E-3 * r1 * q1, 0.1346) * S.s[S_PRECIP_FAC]);
    const double rain = -r1 * (0.5 * (at(S.w, G, i, 2) + 0.) - VT) * q1;
    S.precip[i] = (rain < 0) ? 0. : rain;
}

// BoundaryProcess2D_center (westdown = 0) or _westdown on one field.
__global__ void __launch_bounds__(BX *BY) k_bc_one(Grid G, double *a, int westdown) {
    const int i = blockIdx.x * BX + threadIdx.x, k = blockIdx.y * BY + uniform(threadIdx.y);
    if (i >= G.nx || k >= G.nz) return;
    if (westdown) bc_westdown_cell(a, G, i, k);
    else bc_center_cell(a, G, i, k);
}

__global__ void __launch_bounds__(1024) k_pubartop(Grid G, StepPtrs S, int step) { pubartop_block(G, S, step); }

inline dim3 grid2d(const Grid &G) { return dim3((G.nx + BX - 1) / BX, (G.nz + BY - 1) / BY); }
// tiles from the first interior point on (2048 x 256: 2048 of them, one round
// at eight workgroups a CU; from the ghost cells on, 2145)
inline dim3 interior_grid(const Grid &G) { return dim3((G.nx - 2 + BX - 1) / BX, (G.nz - 2 + BY - 1) / BY); }

}  // namespace

void launch_pzeta(const Grid &G, const StepPtrs &S, int step, hipStream_t st) {
    const dim3 g = xcd_grid(pz_tiles_x(G) * pz_tiles_z(G));
    if (past_caches(G)) hipLaunchKernelGGL((k_pzeta<PZ_BOTH, true>), g, dim3(PZX, PZY), 0, st, G, S, step);
    else hipLaunchKernelGGL((k_pzeta<PZ_BOTH, false>), g, dim3(PZX, PZY), 0, st, G, S, step);
}
void launch_advection_zeta(const Grid &G, const StepPtrs &S, int step, hipStream_t st) {
    const dim3 g = xcd_grid(pz_tiles_x(G) * pz_tiles_z(G));
    hipLaunchKernelGGL(k_pzeta<PZ_ADV>, g, dim3(PZX, PZY), 0, st, G, S, step);
}
void launch_buoyancy(const Grid &G, const StepPtrs &S, int step, hipStream_t st) {
    const dim3 g = xcd_grid(pz_tiles_x(G) * pz_tiles_z(G));
    hipLaunchKernelGGL(k_pzeta<PZ_BUOY>, g, dim3(PZX, PZY), 0, st, G, S, step);
}
void launch_advection_scalar(const Grid &G, const StepPtrs &S, int step, int field, hipStream_t st) {
    hipLaunchKernelGGL(k_adv_scalar, grid2d(G), dim3(BX, BY), 0, st, G, S, step, field);
}
void launch_advection_qrvt(const Grid &G, const StepPtrs &S, int step, hipStream_t st) {
    hipLaunchKernelGGL(k_qrvt, grid2d(G), dim3(BX, BY), 0, st, G, S, step);
}
void launch_precip(const Grid &G, const StepPtrs &S, hipStream_t st) {
    hipLaunchKernelGGL(k_precip, dim3((G.nx + 255) / 256), dim3(256), 0, st, G, S);
}
void launch_bc_one(const Grid &G, double *a, bool westdown, hipStream_t st) {
    hipLaunchKernelGGL(k_bc_one, grid2d(G), dim3(BX, BY), 0, st, G, a, int(westdown));
}
Negval launch_thermo4(const Grid &G, const StepPtrs &S, int step, const RedSlot &rs, hipStream_t st) {
    const int n = advect_tiles(G);
    if (past_caches(G)) hipLaunchKernelGGL(k_thermo4<true>, xcd_grid(n), dim3(T4X, T4Y), 0, st, G, S, step, rs);
    else hipLaunchKernelGGL(k_thermo4<false>, xcd_grid(n), dim3(T4X, T4Y), 0, st, G, S, step, rs);
    return {rs, n};
}
int advect_tiles(const Grid &G) { return t4_tiles_x(G) * t4_tiles_z(G); }
// Up to 1024 tiles of each, four to a CU and one round: there the two shorten
// each other's last round and save a launch.  On large grids the launch is
// nothing and thermo4's LDS keeps CUs from filling up with pzeta's tiles.  A
// step in us, together / apart: 128 x 64 55.7 / 63.5, 1024 x 128 78.9 / 83.1,
// 1536 x 256 128.0 / 132.2, 2048 x 256 (1024 tiles) 142.2 / 143.4; past the line
// the last round decides, 1152 tiles 163.4 / 168.1, 1280 171.5 / 172.8, 1536
// 193.5 / 199.1, 1792 236.5 / 226.7, 2048 (4096 x 256) 252.4 / 235.6: the line is
// the last whole round, not the last grid that gains.
bool advect_together(const Grid &G) { return advect_tiles(G) <= 1024; }
Negval launch_advect(const Grid &G, const StepPtrs &S, int step, const RedSlot &rs, hipStream_t st) {
    const int n = advect_tiles(G);  // no fewer than pzeta's
    hipLaunchKernelGGL(k_advect, xcd_grid(2 * n), dim3(T4X, T4Y), 0, st, G, S, step, rs);
    return {rs, n};
}
// The ratios of NegativeValueProcess from nblk workgroups' partials: by
// k_finalize (nblk 0 is returned), or, up to kFoldBlocks, by the workgroups of
// the second pass themselves (nblk).  The launch costs 4 to 5 us
// whatever it does; every workgroup's own sum costs the traffic of all partials
// for each of them, which at 2048 x 256 (1024 partials of thermo4, 2048 of
// k_kessler) is no gain.
Negval negval_partials(const StepPtrs &S, const Negval &nv, hipStream_t st) {
    if (nv.nblk <= kFoldBlocks) return nv;
    finalize<6>(nv.rs, nv.nblk, S.s, RED_NEGVAL, S_NEG_RATIO, st);
    return {nv.rs, 0};
}
void launch_scale_forcing(const Grid &G, const StepPtrs &S, const Negval &nv, const Forcing &F, hipStream_t st,
                          bool halos) {
    hipLaunchKernelGGL(k_scale_forcing, interior_grid(G), dim3(BX, BY), 0, st, G, S, nv, F, int(halos));
}
void launch_bc_uw(const Grid &G, const StepPtrs &S, hipStream_t st) {
    hipLaunchKernelGGL(k_bc_uw, grid2d(G), dim3(BX, BY), 0, st, G, S);
}
void launch_bc_all_prog(const Grid &G, const StepPtrs &S, hipStream_t st) {
    hipLaunchKernelGGL(k_bc_all, grid2d(G), dim3(BX, BY), 0, st, G, S);
}
void launch_pubartop(const Grid &G, const StepPtrs &S, int step, hipStream_t st) {
    hipLaunchKernelGGL(k_pubartop, dim3(1), dim3(1024), 0, st, G, S, step);
}

}  // namespace vvmd
