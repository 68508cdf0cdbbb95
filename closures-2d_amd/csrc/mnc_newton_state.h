// mnc_newton_state.h -- what the Newton kernels share: the per-cell state in
// HBM, the regularization ladder, the tests that every form of the per-cell
// logic applies (opt.cpp:154-343) and the tail's work list.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>

#include "mnc_internal.h"

namespace mnc {
namespace {

#define kSqrtPi sqrt(M_PI)
#define kPi M_PI
__constant__ double kReg[5] = {0.0, 1e-3, 1e-2, 1e-1, 5e-1};   // opt.h:39-40
enum : int { ST_NEWTON = 0, ST_TRIAL = 1 };

// ---- per-cell solver state in HBM ------------------------------------------
// Structure of arrays [field][cap]: threads handling neighbouring list entries
// (mostly ascending cell indices) touch neighbouring words.
// Moment order N of n = (N+1)(N+2)/2 moments, and the order-2N count padded to
// the 16 columns of an MFMA tile (the mixed sweep's Hessian moments).
constexpr int order_of(int nm) { int N = 0; while ((N + 1) * (N + 2) / 2 < nm) ++N; return N; }
constexpr int mix_cols(int nm) { return ((2 * order_of(nm) + 1) * (2 * order_of(nm) + 2) / 2 + 15) / 16 * 16; }
constexpr int cmax(int a, int b) { return a > b ? a : b; }

template <int NM, int NP2>
struct Store {
    static constexpr int nacc = cmax(cmax(NP2, NM * (NM + 1) / 2), mix_cols(NM));
    enum : int {
        F_AL = 0, F_U = NM, F_AOLD = 2 * NM, F_D = 3 * NM, F_T = 4 * NM, F_RTOL, F_U0, F_ASCALE, F_FCUR,
        F_GD, F_MAXF, F_FSCALE, F_DELTA, F_SF, F_GS, F_ACC = F_GS + NM
    };
    static constexpr int dfields = F_ACC + nacc;
    enum : int { I_ITER = 0, I_TOTAL, I_REG, I_MAXIT, I_MODE, I_WARM, ifields };
    double *D;
    int *I;
    size_t cap;
    __device__ double &d(int f, int c) const { return D[size_t(f) * cap + c]; }
    __device__ int &i(int f, int c) const { return I[size_t(f) * cap + c]; }
};

// The supplementary stop test (opt.cpp:52-76,288-293): with tol_gamma > 0 a
// cell whose gradient passes the tolerance stops only when
// gamma = exp(2 |d|_1 m_inf) (Mn) or 1 + 2 |d|_1 m_inf (PPn) is <= tol_gamma,
// d the Newton direction and m_inf = sqrt((2 P + 1) / (2 pi)) with
// P = floor(sqrt(n)) + 1 (computed on the host).  da1 is |d|_1 summed in
// index order.
__device__ __forceinline__ bool gamma_ok(const NewtonArgs &A, double da1, bool ppn) {
    const double x = 2.0 * da1 * A.gamma_minf;
    return (ppn ? 1.0 + x : exp(x)) <= A.tol_gamma;
}

// The learned warm start's fallback: a cell started from the network's guess
// (I_WARM 0) that meets a regularization criterion at level 0 -- the iteration
// limit, a failed factorisation, an exhausted line search, a condition estimate
// above cond_h_max -- within A.fallback_iters Newton iterations restarts once
// from isotropicAlpha at level 0 instead of climbing the ladder: the guess, not
// the problem, may be what failed, and the start from isotropicAlpha is the
// reference's own (momopt_update.cpp:236-238 with an isotropic previous alpha).
// A late failure is the problem's (cells beyond what the quadrature resolves
// fail at level 0 from any start) and climbs the ladder.  I_WARM becomes
// kWarmFellBack, so a second failure climbs the ladder as the reference does.
// Only Mn, where the network exists.
constexpr int kWarmFellBack = 3;
__device__ __forceinline__ bool net_fallback(const NewtonArgs &A, int reg, int warm, int iter) {
    return reg == 0 && warm == 0 && iter <= A.fallback_iters;
}

// The PPn ansatz at t = (alpha.m)/2 (fobj.cpp:166-172): G = t + s with
// s = sqrt(t^2 + delta), taken as -delta / (t - s) for t < 0.
__device__ __forceinline__ double ppn_g(double t, double delta, double &s) {
    s = sqrt(t * t + delta);
    return t < 0.0 ? -delta / (t - s) : t + s;
}

// Control word holding the count of list l: lists 0 and 1 (the lockstep
// ping-pong pair) use words 0 and 1, lists 2 and 3 (the FP64 pair of a
// mixed-precision solve) words 4 and 5, list 4 (the learned warm start's
// network rows) word 6.  Word 2 is the tail's queue head, word 3 the error bits.
__device__ __forceinline__ int cw(int l) { return l < 2 ? l : l + 2; }

// Entry s of the tail's work: the cells left on list `lin`, then those left
// on list `lin2` (the FP64 list of a mixed-precision solve).  -1 past the end.
__device__ __forceinline__ int tail_cell(const NewtonArgs &A, int lin, int count, int lin2, int count2, int s) {
    if (s < count) return A.lists[size_t(lin) * A.cap + s];
    if (s < count + count2) return A.lists[size_t(lin2) * A.cap + (s - count)];
    return -1;
}

}  // namespace
}  // namespace mnc
