// direct.h -- the cal_w system L x = f by a direct method (k_direct.hip).
//
// L has constant coefficients along the periodic x, so the discrete Hartley
// transform along x (real, its own inverse up to 1/N) makes it one tridiagonal
// system along z for each of the N frequencies: diagonal
// cx_j lambda_q + cu_j + cu_{j-1}, lambda_q = 4 sin^2(pi q / N), off-diagonal
// -cu_j.  Any N and M: the transform is a mixed-radix FFT (8, 4, 2, 3, 5, and
// direct sums for small other prime factors); with large ones a convolution.
#pragma once

#include "vvm_internal.h"

namespace vvmd {

struct Micro;

constexpr int kMaxStages = 16;

// The factors of L and the launch shape of the row transforms.
struct RowPlan {
    int N = 0, M = 0;
    int L = 0;            // the FFT's length: N, or the convolution's (chirp)
    int chirp = 0;        // large prime factors: the transform as a convolution
    int nst = 0, radix[kMaxStages] = {};
    int threads = 0;      // at least L / 8: a thread holds at most 8 outputs of a stage
    // in LDS: nothing, the table of all roots (a prime factor above 5 reads it),
    // or the stages' twiddles; nothing where that would pass the LDS size
    enum { TW_GLOBAL, TW_ROOTS, TW_STAGES };
    int tw = TW_GLOBAL;
};

template <typename T>
class Direct {
   public:
    // cx [M+2], cu [M+1]: level-0 coefficients on the device.  Returns VVM_OK
    // or VVM_ERR_NOMEM / VVM_ERR_HIP.
    int init(int N, int M, const double *cx, const double *cu);
    void destroy();
    bool ready() const { return spec != nullptr; }

    // x = L^-1 r on rows 1..M of (M+2) x N arrays, or x0 + L^-1 r if x0 is set
    // (which may be x).
    void solve(const double *r, const double *x0, double *x, hipStream_t st);
    // x = x0 + L^-1 r, and w = x / rhow with its halos.
    void solve_w(const double *r, const double *x0, double *x, const Grid &G, double *w, const double *rhow,
                 hipStream_t st);
    // cal_w whole: f = -b / rhow from zetap (f is written, for the residual),
    // x = L^-1 f, w = x / rhow with its halos; pubarTop_pt beside the first
    // kernel's row transforms (step < 0: not), and the microphysics (if set)
    // beside the first two kernels.
    void solve_step(const Grid &G, const StepPtrs &S, int step, const Micro *micro, double *f, double *x,
                    hipStream_t st);

   private:
    RowPlan plan;
    size_t row_lds = 0, col_lds = 0;
    T *tw = nullptr;    // [L][2]: cos, -sin of 2 pi k / L; then the stages' twiddles, [L-1][2]
    T *chirp = nullptr; // [N][2] the chirp, [L][2] the transform of its inverse, over L
    T *di = nullptr;    // [M][N/2+1] 1 / pivot
    const double *cu_dev = nullptr;
    T *spec = nullptr;  // [M][N] transformed rows
    template <bool C>
    void rows_solve(const double *r, const double *x0, double *x, const Grid &G, double *w, const double *rhow,
                    hipStream_t st);
    template <bool C>
    void rows_solve_step(const Grid &G, const StepPtrs &S, int step, const Micro *micro, double *f, double *x,
                         hipStream_t st);
    template <typename Mic>
    void columns(const Mic &mic, int nmic, hipStream_t st);
};

}  // namespace vvmd
