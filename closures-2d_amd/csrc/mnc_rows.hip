// mnc_rows.hip -- the FP64 Newton solve with a 16-lane row per cell.
//
// A wave carries four cells, one per 16-lane DPP row, or (WIDE) one cell, and
// iterates each to completion from a queue: the whole per-cell algorithm
// (opt.cpp:82-343, linesearch.cpp:21-99, fobj.cpp:37-129,255-335) in one
// launch, with no per-cell state in HBM.
//
// An evaluation has two layouts.
//  Sweep: lanes 4c..4c+3 of every 16-lane row work for cell c on the orbits
//   o = slot, slot + 16, ... of the quadrature (mnc_orbit.h); WIDE: all 64
//   lanes work for the one cell.  A lane forms the four exponents of an orbit
//   from one pass over its moments, combines w e into the four class sums
//   C[c], and accumulates the Hessian sums class by class (at most 40 of the
//   120 sums of n = 15 are live at once, so that two waves fit a SIMD).  Each
//   class's sums are reduced over the sixteen lanes of a cell in four exchange
//   steps that halve the values a lane holds (v_permlane32/16_swap across the
//   rows, quad permutations within), and stored to LDS.
//  Algebra: lane r of row c holds row r of cell c's H.  The Cholesky factor,
//   L^-1 (lane j its column j, lane n the gradient beside them), the Newton
//   direction L^-T (L^-1 g) and the condition bounds broadcast one lane's
//   value to its row (DPP row_newbcast), so the four cells' dependent steps
//   run side by side and nothing goes through LDS.
// What bounds it: FP64 issue and the dependent steps of the algebra.  Two waves per
// SIMD leave 256 registers, which the M4 forms of Mn exceed by 20 (four cells per
// wave) and 16; PPn and the lower orders fit.  With the cell's state in registers,
// the factor's 105 broadcasts kept for the inverse and a branch around each load of H
// they exceeded them by 316, and scratch traffic was three quarters of the time
// (150,001 closures 7.0 ms a call, now 2.85).  Further times stand at the launch rule
// (launch_rows_n).
#include <cfloat>

#include "mnc_newton_state.h"
#include "mnc_coop_la.h"
#include "mnc_orbit.h"

namespace mnc {
namespace {

template <int I> struct Int { static constexpr int value = I; };
template <int B, int E, class F>
__device__ __forceinline__ void unroll(F &&f) {
    if constexpr (B < E) {
        f(Int<B>{});
        unroll<B + 1, E>(f);
    }
}

// lane K of each 16-lane row, on every lane of the row
template <int K>
__device__ __forceinline__ double row_bcast(double v) {
    return __builtin_amdgcn_update_dpp(0.0, v, 0x150 + K, 0xf, 0xf, true);
}
// Sum over the 16 lanes of a row, the same bits on every lane (the decisions
// taken from it are row-uniform): each step adds two partial sums that a pair
// of lanes exchanges -- quad permutations, then the mirror images within 8
// and 16 lanes.  Rotations would add the quads in another order on each lane,
// and a caller's product contracted into the first addition would be rounded
// on one lane of a pair and not on the other: the empty asm takes the value
// as rounded.
__device__ __forceinline__ double row_sum(double v) {
    __asm__("" : "+v"(v));
    v += dpp_row_d<0xB1>(v);
    v += dpp_row_d<0x4E>(v);
    v += dpp_row_d<0x141>(v);
    v += dpp_row_d<0x140>(v);
    return v;
}
// max and min over the 16 lanes of a row, on every lane (they do not round)
__device__ __forceinline__ double row_max(double v) {
    v = fmax(v, dpp_row_d<0xB1>(v));
    v = fmax(v, dpp_row_d<0x4E>(v));
    v = fmax(v, dpp_row_d<0x124>(v));
    v = fmax(v, dpp_row_d<0x128>(v));
    return v;
}
__device__ __forceinline__ double row_min(double v) {
    v = fmin(v, dpp_row_d<0xB1>(v));
    v = fmin(v, dpp_row_d<0x4E>(v));
    v = fmin(v, dpp_row_d<0x124>(v));
    v = fmin(v, dpp_row_d<0x128>(v));
    return v;
}

// Half of each of two values' lanes exchanged: lanes of the lower half (of
// the even rows for swap16) leave with x summed over the pair of lanes, the
// others with y.
__device__ __forceinline__ double swap32_add(double x, double y) {
    const unsigned long long a = (unsigned long long)__double_as_longlong(x), b = (unsigned long long)__double_as_longlong(y);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)a, (unsigned)b, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(a >> 32), (unsigned)(b >> 32), false, false);
    return __longlong_as_double((long long)((unsigned long long)hi[0] << 32 | lo[0])) +
           __longlong_as_double((long long)((unsigned long long)hi[1] << 32 | lo[1]));
}
__device__ __forceinline__ double swap16_add(double x, double y) {
    const unsigned long long a = (unsigned long long)__double_as_longlong(x), b = (unsigned long long)__double_as_longlong(y);
    const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)a, (unsigned)b, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(a >> 32), (unsigned)(b >> 32), false, false);
    return __longlong_as_double((long long)((unsigned long long)hi[0] << 32 | lo[0])) +
           __longlong_as_double((long long)((unsigned long long)hi[1] << 32 | lo[1]));
}

// v[0..V-1] summed over the sixteen lanes of a cell (lane bits 0, 1, 4, 5)
// into out[0..V-1] of that cell: each step keeps half of the values, the bits
// of the lane say which.  add: onto what out holds.
template <int V>
__device__ __forceinline__ void reduce_store(const double (&v)[V], double *out, int lane, bool add) {
    constexpr int A = (V + 1) / 2, B = (A + 1) / 2, C = (B + 1) / 2, D = (C + 1) / 2;
    double a[A], b[B], c[C];
#pragma unroll
    for (int r = 0; r < A; ++r) a[r] = swap32_add(v[r], A + r < V ? v[A + r] : 0.0);
#pragma unroll
    for (int r = 0; r < B; ++r) b[r] = swap16_add(a[r], B + r < A ? a[B + r] : 0.0);
    const bool b0 = lane & 1, b1 = lane & 2;
#pragma unroll
    for (int r = 0; r < C; ++r) {
        const double lo = b[r], hi = C + r < B ? b[C + r] : 0.0;
        c[r] = (b0 ? hi : lo) + dpp_row_d<0xB1>(b0 ? lo : hi);
    }
    const int at = (lane & 32 ? A : 0) + (lane & 16 ? B : 0) + (b0 ? C : 0) + (b1 ? D : 0);
#pragma unroll
    for (int r = 0; r < D; ++r) {
        const double lo = c[r], hi = D + r < C ? c[D + r] : 0.0;
        const double s = (b1 ? hi : lo) + dpp_row_d<0x4E>(b1 ? lo : hi);
        const int i3 = (b1 ? D : 0) + r, i2 = (b0 ? C : 0) + i3, i1 = (lane & 16 ? B : 0) + i2;
        if (i3 < C && i2 < B && i1 < A && at + r < V) {
            if (add) out[at + r] += s;
            else out[at + r] = s;
        }
    }
}

// x <- (L L^T)^{-1} x with x_i on lane i of the row: row holds L's row, col
// its column below the diagonal, rd[j] = 1 / L_jj.
template <int NM>
__device__ __forceinline__ void rows_apply_inv(const double (&row)[NM], const double (&col)[NM],
                                               const double (&rd)[NM], double &x, int r) {
    unroll<0, NM>([&](auto J) {
        constexpr int j = decltype(J)::value;
        const double xj = row_bcast<j>(x) * rd[j];
        x = r == j ? xj : (r > j && r < NM ? fma(-xj, row[j], x) : x);
    });
    unroll<0, NM>([&](auto J) {
        constexpr int j = NM - 1 - decltype(J)::value;
        const double xj = row_bcast<j>(x) * rd[j];
        x = r == j ? xj : (r < j ? fma(-col[j], xj, x) : x);
    });
}

// Reciprocal 1-norm condition estimate per row (Higham 1988, dpocon's role).
template <int NM>
__device__ __forceinline__ double rows_rcond(const double (&row)[NM], const double (&col)[NM], const double (&rd)[NM],
                                             double anorm, int lane) {
    const int r = lane & 15;
    const int shift = lane & 48;
    unsigned isgn = 0;
    double est = 0.0;
    int jump = 1, j = 0, iter = 0;
    double x = r < NM ? 1.0 / NM : 0.0;
#pragma unroll 1
    for (int guard = 0; guard < 16 && jump != 0; ++guard) {
        rows_apply_inv<NM>(row, col, rd, x, r);
        const double v = r < NM ? fabs(x) : -1.0;
        const double s = row_sum(r < NM ? v : 0.0);
        const double m = row_max(v);
        const unsigned at = (unsigned)(__ballot(v == m) >> shift) & 0xffffu;
        const int im = at ? __ffs((int)at) - 1 : 0;          // the first largest (idamax)
        const unsigned sg = (unsigned)(__ballot(r < NM && !(x >= 0.0)) >> shift) & 0xffffu;
        const double xj = __shfl(x, shift + j);
        double nx = 0.0;
        if (jump == 1) {
            if (NM == 1) { est = s; jump = 0; }
            else { est = s; isgn = sg; nx = (sg >> r & 1u) ? -1.0 : 1.0; jump = 2; }
        } else if (jump == 2) {
            j = im; iter = 2; nx = r == j ? 1.0 : 0.0; jump = 3;
        } else if (jump == 3) {
            const double estold = est;
            est = s;
            if (sg == isgn || est <= estold) {
                nx = ((r & 1) ? -1.0 : 1.0) * (1.0 + double(r) / double(NM - 1));
                jump = 5;
            } else {
                nx = (sg >> r & 1u) ? -1.0 : 1.0;
                isgn = sg;
                jump = 4;
            }
        } else if (jump == 4) {
            j = im;
            if (xj != m && iter < 5) {
                ++iter; nx = r == j ? 1.0 : 0.0; jump = 3;
            } else {
                nx = ((r & 1) ? -1.0 : 1.0) * (1.0 + double(r) / double(NM - 1));
                jump = 5;
            }
        } else {
            const double temp = 2.0 * (s / double(3 * NM));
            if (temp > est) est = temp;
            jump = 0;
        }
        x = r < NM ? nx : 0.0;
    }
    if (anorm == 0.0 || !isfinite(est) || est == 0.0) return 0.0;
    return (1.0 / est) / anorm;
}

constexpr int kRowWaves = 4;      // waves per block
constexpr int kRowTiles = 4;      // orbit tiles whose class sums are kept in registers (four cells per wave)

// What a cell carries from one evaluation to the next, in LDS beside the wave's
// sums: in registers it would stand beside the sums and the factor, and spill.
enum : int { V_UL, V_AOLD, V_DL, kRowVectors };                  // an element per lane
enum : int { S_U0, S_ASCALE, S_RTOL, S_FCUR, S_GD, S_FSCALE, S_MAXF, S_DELTA, kRowScalars };   // one per row
// Counts of a row (its lane 0 counts).
enum : int { R_MAX_ITER, R_ERR, R_SUM, R_N, R_TRIALS, R_HIST, R_CELLS = R_HIST + 5, R_TITER, R_FALLBACK, R_ISO, R_PREV,
             kRowCounts };

template <int N, bool GAUNT, bool PPN, bool WIDE>
struct RowDims {
    static constexpr int NM = orbit_nm(N), NP2 = GAUNT ? orbit_nm(2 * N) : NM;
    static constexpr int NS = OrbitSums<N, GAUNT>::count;
    static constexpr int RAW = NS + 1 + (PPN ? NM : 0);           // sums per cell in LDS
    static constexpr int RAWP = RAW | 1;
    // per wave: the sums, the iterates, the cells' state, the counts
    static constexpr int LANE_WORDS = 4 * RAWP + 64 + 64 * kRowVectors + 4 * kRowScalars + 2 * kRowCounts;
    static constexpr int TB = WIDE ? 1 : kRowTiles;
};

// The cells of [0, ncells) from their u and alpha (fresh), or the cells left
// on lists lin and lin2 from their state in HBM.  few: the host launched both
// kernels without knowing the lists' counts; with at most one cell per wave
// the WIDE one runs and the other leaves at once, else the other way round.
template <int N, bool GAUNT, bool PPN, bool WIDE, bool TABLED>
__global__ __launch_bounds__(64 * kRowWaves) __attribute__((amdgpu_waves_per_eu(2)))
void rows_kernel(NewtonArgs A, int lin, int lin2, int fresh, int few) {
    using Dm = RowDims<N, GAUNT, PPN, WIDE>;
    constexpr int NM = Dm::NM, NP2 = Dm::NP2, NS = Dm::NS, RAWP = Dm::RAWP, TB = Dm::TB;
    constexpr int SLOTS = WIDE ? 64 : 16;
    using St = Store<NM, NP2>;
    using Sums = OrbitSums<N, GAUNT>;
    constexpr typename Sums::Lists L = Sums::lists();
    extern __shared__ double lds[];
    __shared__ int red[kRowWaves][16];
    int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // its LDS addresses in scalar registers
    const int count = fresh ? A.ncells : A.ctl[cw(lin)];
    const int total_cells = count + (fresh ? 0 : A.ctl[cw(lin2)]);
    const int waves = gridDim.x * kRowWaves;
    if (total_cells == 0 || (few != 0 && (total_cells <= waves) != WIDE)) return;   // uniform
    const int tiles = (A.no + SLOTS - 1) / SLOTS;
    constexpr int TILE = (NP2 + 1) * 16;                        // table words of 16 orbits: [k][16], weights last
    const int table = TABLED ? A.nop / 16 * TILE : 0;
    if constexpr (TABLED) {
        for (int i = threadIdx.x; i < table; i += blockDim.x) lds[i] = A.ot[i];
    }
    double *raw = lds + table + wave * Dm::LANE_WORDS, *als = raw + 4 * RAWP;
    double *vectors = als + 64, *scalars = vectors + 64 * kRowVectors;
    int *counts = reinterpret_cast<int *>(scalars + 4 * kRowScalars);
    for (int i = lane; i < 64 * kRowVectors + 4 * kRowScalars + 2 * kRowCounts; i += 64) vectors[i] = 0.0;
    __syncthreads();
    const double p0 = A.p[0];
    const int per_wave = WIDE ? 1 : min(4, max(1, (total_cells + waves - 1) / waves));
    // per-cell state beside the one in LDS: the iterate one element per lane, scalars on every lane of the row
    int c = (!WIDE && (lane >> 4) >= per_wave) ? -2 : -1;              // -1 wants a cell, -2 has none left to take
    double al = 0.0, t = 1.0;
    int mode = ST_NEWTON, iter = 0, total = 0, reg = 0, maxit = 0, warm = 2;
    for (;;) {
        // the lane's masks and offsets are formed anew each pass: kept across
        // the loop they would take the registers the sums need
        __asm__ volatile("" : "+v"(lane));
        const int r = lane & 15, rowc = lane >> 4;              // algebra: row r of cell rowc
        const int cj = (lane >> 2) & 3;                         // sweep: cell cj, orbit slot
        const int slot = WIDE ? (lane >> 4) * TILE + (lane & 15) : (lane & 3) | (rowc << 2);
        const bool owner = WIDE ? rowc == 0 : true;             // WIDE: the four rows repeat one cell
        const bool in = r < NM;
        double *myraw = raw + (WIDE ? 0 : rowc * RAWP);
        double *vl = vectors + lane, *sr = scalars + rowc;
        int *st = counts + rowc * kRowCounts;
        // ---- cells for the rows without one ----
        const unsigned long long want = WIDE ? (__ballot(c == -1) & 1ull) : __ballot(c == -1 && r == 0);
        if (want) {
            int base = 0;
            if (lane == 0) base = atomicAdd(&A.ctl[2], __popcll(want));
            base = __builtin_amdgcn_readfirstlane(base);
            if (c == -1) {
                const int s = base + (WIDE ? 0 : __popcll(want & ((1ull << (lane & 48)) - 1ull)));
                if (s >= total_cells) {
                    c = -2;
                } else if (fresh) {                             // opt.cpp:87-101,170-205
                    c = s;
                    const double u0 = A.u[size_t(c) * NM], ascale = log(u0) * 2.0 * kSqrtPi;
                    const double ul = in ? A.u[size_t(c) * NM + r] / u0 : 0.0;
                    const double delta = PPN ? A.delta / (u0 * u0) : 0.0;
                    sr[4 * S_U0] = u0;
                    sr[4 * S_ASCALE] = ascale;
                    vl[64 * V_UL] = ul;
                    if constexpr (PPN) sr[4 * S_DELTA] = delta;
                    // isotropicAlpha (opt.cpp:27-46) if asked for, or (the learned
                    // start with its network off) if the alpha passed in is not finite
                    al = in ? A.alpha[size_t(c) * NM + r] : 0.0;
                    bool iso = A.warm == MNC_WARM_ISOTROPIC;
                    if (A.warm == MNC_WARM_LEARNED) {
                        iso = row_max(isfinite(al) ? 0.0 : 1.0) != 0.0;
                        if (owner && r == 0) { st[R_ISO] += iso; st[R_PREV] += !iso; }
                        warm = iso ? 1 : 2;
                    }
                    if (iso) al = r == 0 ? (PPN ? 1.0 - 4.0 * delta * kPi : 2.0 * kSqrtPi * log(0.5 / kSqrtPi)) : 0.0;
                    else if (PPN) al = al / u0;
                    else if (r == 0) al = al - ascale;
                    sr[4 * S_RTOL] = sqrt(row_sum(ul * ul)) * A.tol;
                    t = 1.0;
                    iter = total = reg = 0;
                    maxit = A.max_iter;
                    mode = ST_NEWTON;
                    if (!(u0 > 0.0)) {
                        if (owner && r == 0) {
                            st[R_ERR] |= 1 << MNC_ERR_U0;
                            if (A.outs) { A.outs[c].iter = -1; A.outs[c].r = 0.0; A.outs[c].norm_g = 0.0; }
                        }
                        c = -1;
                    } else if (owner && r == 0) {
                        ++st[R_CELLS];
                    }
                } else {
                    c = s < count ? A.lists[size_t(lin) * A.cap + s] : A.lists[size_t(lin2) * A.cap + (s - count)];
                    const St S{A.st_d, A.st_i, A.cap};
                    al = in ? S.d(St::F_AL + r, c) : 0.0;
                    const double aold = in ? S.d(St::F_AOLD + r, c) : 0.0;
                    vl[64 * V_UL] = in ? S.d(St::F_U + r, c) : 0.0;
                    vl[64 * V_AOLD] = aold;
                    vl[64 * V_DL] = in ? S.d(St::F_D + r, c) : 0.0;
                    t = S.d(St::F_T, c);
                    sr[4 * S_RTOL] = S.d(St::F_RTOL, c);
                    sr[4 * S_U0] = S.d(St::F_U0, c);
                    sr[4 * S_ASCALE] = S.d(St::F_ASCALE, c);
                    sr[4 * S_FCUR] = S.d(St::F_FCUR, c);
                    sr[4 * S_GD] = S.d(St::F_GD, c);
                    sr[4 * S_FSCALE] = S.d(St::F_FSCALE, c);
                    sr[4 * S_MAXF] = S.d(St::F_MAXF, c);
                    if constexpr (PPN) sr[4 * S_DELTA] = S.d(St::F_DELTA, c);
                    mode = S.i(St::I_MODE, c);
                    iter = S.i(St::I_ITER, c);
                    total = S.i(St::I_TOTAL, c);
                    reg = S.i(St::I_REG, c);
                    maxit = S.i(St::I_MAXIT, c);
                    warm = S.i(St::I_WARM, c);
                    if (owner && r == 0) {
                        ++st[R_CELLS];
                        st[R_TITER] -= total;
                    }
                    // The reference's Armijo test compares values of f down to
                    // their rounding, which differs between the kernels: a
                    // search begun elsewhere starts again from its own iterate,
                    // evaluated here (the robust rule has no such need).
                    if (A.ls_mode == MNC_LS_REFERENCE && mode == ST_TRIAL) {
                        al = aold;
                        mode = ST_NEWTON;
                        t = 1.0;
                        --iter;
                        --total;
                    }
                }
            }
        }
        if (__ballot(c >= 0) == 0) {
            if (__ballot(c == -1) == 0) break;
            continue;
        }
        // ---- the sweep ----
        als[r * 4 + rowc] = PPN && r == 15 ? sr[4 * S_DELTA] : al;
        __builtin_amdgcn_wave_barrier();
        // after two failed trials only f is summed: the next trials mostly fail
        // too, and an accepted one is evaluated in full afterwards
        const bool fonly = __ballot(c >= 0 && !(mode == ST_TRIAL && t < 0.3)) == 0;
        for (int t0 = 0; t0 < tiles; t0 += TB) {
            // table word of moment 0 of this lane's orbit in tile t0
            const double *tp = (TABLED ? lds : A.ot) + t0 * (SLOTS / 16) * TILE + slot;
            constexpr int STEP = (SLOTS / 16) * TILE;
            double C[4][TB];
            double gs[PPN ? NM + 1 : 1];
            if constexpr (PPN) {
#pragma unroll
                for (int k = 0; k <= NM; ++k) gs[k] = 0.0;
            }
            {
                double av[NM];
#pragma unroll
                for (int k = 0; k < NM; ++k) av[k] = als[k * 4 + cj];
                const double dj = PPN ? als[15 * 4 + cj] : 0.0;
#pragma unroll
                for (int tt = 0; tt < TB; ++tt) {
                    if (t0 + tt >= tiles) {                      // uniform
                        C[0][tt] = C[1][tt] = C[2][tt] = C[3][tt] = 0.0;
                        continue;
                    }
                    double s[4] = {0.0, 0.0, 0.0, 0.0};
                    double m[NM];
#pragma unroll
                    for (int k = 0; k < NM; ++k) {
                        m[k] = tp[tt * STEP + k * 16];
                        s[L.cls[k]] = fma(av[k], m[k], s[L.cls[k]]);
                    }
                    const double w = tp[tt * STEP + NP2 * 16];
                    const double p = s[0] + s[1], q = s[0] - s[1], u = s[2] + s[3], v = s[2] - s[3];
                    const double z[4] = {p + u, q + v, p - u, q - v};      // ++, -+, +-, --
                    double e[4];
                    if constexpr (PPN) {
                        double G[4], f = 0.0;
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const double tq = 0.5 * z[i];
                            double sq;
                            G[i] = ppn_g(tq, dj, sq);
                            e[i] = 0.5 * (G[i] / sq);
                            f = f + (tq * G[i] - 0.5 * dj + dj * log(G[i]));
                        }
                        gs[NM] += w * f;
                        const double ga = G[0] + G[2], gb = G[1] + G[3], gc = G[0] - G[2], gd = G[1] - G[3];
                        const double cg[4] = {w * (ga + gb), w * (ga - gb), w * (gc + gd), w * (gc - gd)};
#pragma unroll
                        for (int k = 0; k < NM; ++k) gs[k] = fma(cg[L.cls[k]], m[k], gs[k]);
                    } else {
#pragma unroll
                        for (int i = 0; i < 4; ++i) e[i] = exp(z[i]);
                    }
                    const double ea = e[0] + e[2], eb = e[1] + e[3], ec = e[0] - e[2], ed = e[1] - e[3];
                    C[0][tt] = w * (ea + eb);
                    C[1][tt] = w * (ea - eb);
                    C[2][tt] = w * (ec + ed);
                    C[3][tt] = w * (ec - ed);
                    __builtin_amdgcn_sched_barrier(0);           // one tile's chains at a time
                }
            }
            double *out = raw + cj * RAWP;
            if constexpr (PPN) reduce_store<NM + 1>(gs, out + NS, lane, t0 > 0);
            if (fonly) {
                if constexpr (!PPN) {
                    double f[1] = {0.0};
#pragma unroll
                    for (int tt = 0; tt < TB; ++tt) f[0] += C[0][tt];
                    reduce_store<1>(f, out + L.first[1], lane, t0 > 0);
                }
            } else {
                unroll<0, 4>([&](auto CC) {
                    constexpr int cc = decltype(CC)::value;
                    constexpr int E0 = L.first[cc], E1 = L.first[cc + 1];
                    constexpr int SF = (!PPN && cc == 0) ? 1 : 0;
                    if constexpr (E1 - E0 + SF > 0) {
                        double acc[E1 - E0 + SF];
#pragma unroll
                        for (int e = 0; e < E1 - E0 + SF; ++e) acc[e] = 0.0;
#pragma unroll
                        for (int tt = 0; tt < TB; ++tt) {
                            if (t0 + tt >= tiles) break;         // uniform
                            const double cw_ = C[cc][tt];
                            if constexpr (SF != 0) acc[E1 - E0] += cw_;
                            if constexpr (GAUNT) {
#pragma unroll
                                for (int e = E0; e < E1; ++e) acc[e - E0] = fma(cw_, tp[tt * STEP + L.a[e] * 16], acc[e - E0]);
                            } else {
                                double m[NM];
#pragma unroll
                                for (int k = 0; k < NM; ++k) m[k] = tp[tt * STEP + k * 16];
                                double v = 0.0;
#pragma unroll
                                for (int e = E0; e < E1; ++e) {
                                    if (e == E0 || L.a[e] != L.a[e > E0 ? e - 1 : e]) v = cw_ * m[L.a[e]];
                                    acc[e - E0] = fma(v, m[L.b[e]], acc[e - E0]);
                                }
                            }
                            // the next tile's rows are not loaded while this one's are live
                            __builtin_amdgcn_sched_barrier(0);
                        }
                        reduce_store<E1 - E0 + SF>(acc, out + orbit_slot(E0, cc, PPN), lane, t0 > 0);
                    }
                });
            }
        }
        __builtin_amdgcn_wave_barrier();
        auto sum_at = [&](int i) -> double {
            if constexpr (WIDE) return (myraw[i] + myraw[RAWP + i]) + (myraw[2 * RAWP + i] + myraw[3 * RAWP + i]);
            else return myraw[i];
        };
        // ---- one step of the per-cell logic ----
        bool done = false;
        if (c >= 0) {
            const double ul = vl[64 * V_UL];
            constexpr int SFP = PPN ? NS + NM : L.first[1];
            const double sf = sum_at(SFP);
            bool newton = mode == ST_NEWTON, do_reg = false, converged = false;
            double err = 0.0, gv = 0.0;
            if (mode == ST_TRIAL) {                             // linesearch.cpp:45-98
                if (owner && r == 0) ++st[R_TRIALS];
                const double fnew = sf - row_sum(al * ul);
                const double gd_s = sr[4 * S_GD];
                bool accept = fnew <= sr[4 * S_FCUR] + 1e-3 * t * gd_s;
                // Robust mode: a full Newton step whose predicted decrease lies
                // below the rounding resolution of f is taken.
                if (!accept && A.ls_mode == MNC_LS_ROBUST && t == 1.0 && -gd_s <= 1e3 * DBL_EPSILON * sr[4 * S_FSCALE])
                    accept = true;
                if (accept) {
                    if (fonly) mode = ST_NEWTON;                // evaluated in full next
                    else newton = true;
                } else {
                    t = 0.5 * t;
                    const double aold = vl[64 * V_AOLD];
                    if (t * sr[4 * S_MAXF] > DBL_EPSILON / 2) {
                        al = fma(t, vl[64 * V_DL], aold);
                    } else {                                    // exhausted
                        al = aold;
                        t = 0.0;
                        ++iter; ++total;
                        do_reg = true;
                    }
                }
            }
            if (newton) {                                       // opt.cpp:212-318
                ++iter; ++total;
                double h[NM];
                if constexpr (GAUNT) {                          // fobj.cpp:99-113
#pragma unroll
                    for (int k = 0; k < NM; ++k) {
                        double hij = 0.0;
                        for (int e = A.ogoff[k]; e < A.ogoff[k + 1]; ++e)
                            hij = fma(A.ogv[e * 16 + r], sum_at(A.ogk[e * 16 + r]), hij);
                        h[k] = hij;
                    }
                } else {
                    unsigned at[4];                             // where H_rk stands among the sums, a byte each
#pragma unroll
                    for (int q = 0; q < 4; ++q) at[q] = reinterpret_cast<const unsigned *>(A.opos)[r * 4 + q];
#pragma unroll
                    for (int k = 0; k < NM; ++k) h[k] = sum_at((at[k >> 2] >> (8 * (k & 3))) & 255u);
                    // every lane loads (row 15 of the places is zeros) before any selects:
                    // as conditional loads these were 15 branches, each with its wait
#pragma unroll
                    for (int k = 0; k < NM; ++k) {
                        __asm__ volatile("" : "+v"(h[k]));
                        h[k] = in ? h[k] : 0.0;
                    }
                }
                const double h00 = row_bcast<0>(h[0]);
                gv = in ? (PPN ? sum_at(NS + r) : h[0] / p0) - ul : 0.0;
                const double au = al * ul;
                double fcur = PPN ? sf : h00 / (p0 * p0);
                const double fscale = fabs(fcur) + row_sum(fabs(au));
                fcur = fcur - row_sum(au);
                double rs = 0.0, dg = 0.0;                      // utils.cpp:36-52
#pragma unroll
                for (int k = 0; k < NM; ++k) {
                    rs += fabs(h[k]);
                    dg = k == r ? h[k] : dg;
                }
                const double anorm = row_max(in ? rs : 0.0);
                const double gersh = row_min(in ? 2.0 * dg - rs : DBL_MAX);
                err = sqrt(row_sum(gv * gv));
                // Cholesky, right-looking (each element sees the subtractions in
                // dpotf2's order); 1 / sqrt of the pivot by v_rsq_f64 and one
                // third-order correction
                bool ok = true;
                double rd[NM];
                unroll<0, NM>([&](auto J) {
                    constexpr int j = decltype(J)::value;
                    double piv = row_bcast<j>(h[j]);
                    ok = ok && piv > 0.0;
                    piv = piv > 0.0 ? piv : 1.0;
                    double x = __builtin_amdgcn_rsq(piv);
                    const double e = fma(-piv * x, x, 1.0);
                    x = fma(x * e, fma(e, 0.375, 0.5), x);
                    rd[j] = x;
                    const double l = h[j] * x;
                    h[j] = l;
                    unroll<j + 1, NM>([&](auto K) {
                        constexpr int k = decltype(K)::value;
                        h[k] = fma(-row_bcast<k>(l), l, h[k]);
                    });
                });
                // the factor as new values: else its 105 broadcasts are kept from the
                // steps above for the ones below, in scratch
#pragma unroll
                for (int k = 0; k < NM; ++k) __asm__ volatile("" : "+v"(h[k]));
                // Z = L^-1, column j on lane j, and L^-1 g on lane NM
                double z[NM];
                unroll<0, NM>([&](auto I) {
                    constexpr int i = decltype(I)::value;
                    const double gi = row_bcast<i>(gv);
                    z[i] = r == NM ? gi : (r == i ? 1.0 : 0.0);
                });
                unroll<0, NM>([&](auto K) {
                    constexpr int k = decltype(K)::value;
                    z[k] = z[k] * rd[k];
                    unroll<k + 1, NM>([&](auto I) {
                        constexpr int i = decltype(I)::value;
                        z[i] = fma(-row_bcast<i>(h[k]), z[k], z[i]);
                    });
                });
                // the direction Z^T (Z g); zero above the diagonal
                double x = 0.0;
                unroll<0, NM>([&](auto K) {
                    constexpr int k = decltype(K)::value;
                    x = fma(row_bcast<NM>(z[k]), z[k], x);
                });
                double condest = 0.0;
                bool ask = ok && !cond_proven_below(anorm, gersh, NM, A.cond_h_max);
                if (ask) {
                    // ||A^-1||_1 <= sqrt(n) trace(A^-1), the trace the sum of Z's squares:
                    // a row's sum against the columns' products below
                    double s = 0.0;
#pragma unroll
                    for (int k = 0; k < NM; ++k) s = fma(z[k], z[k], s);
                    ask = !(2.0 * anorm * sqrt(double(NM)) * row_sum(in ? s : 0.0) <= A.cond_h_max);
                }
                if (ask) {
                    // ||A^-1||_1 from the columns of Z^T Z; the estimate never exceeds it
                    double s = 0.0;
                    unroll<0, NM>([&](auto I) {
                        constexpr int i = decltype(I)::value;
                        double d = 0.0;
                        unroll<i, NM>([&](auto K) {
                            constexpr int k = decltype(K)::value;
                            d = fma(row_bcast<i>(z[k]), z[k], d);
                        });
                        s += fabs(d);
                    });
                    const double inv1 = row_max(in ? s : 0.0);
                    ask = !(2.0 * anorm * inv1 <= A.cond_h_max);
                    if (ask) {
                        // the factor's columns for the back substitutions, through
                        // the cell's own sums (read for the last time above)
                        double col[NM];
#pragma unroll
                        for (int i = 0; i < NM; ++i) col[i] = 0.0;
                        unroll<0, NM>([&](auto K) {
                            constexpr int k = decltype(K)::value;
                            if (owner && in) myraw[r] = h[k];   // column k of L
                            __builtin_amdgcn_wave_barrier();
#pragma unroll
                            for (int i = k + 1; i < NM; ++i) col[i] = r == k ? myraw[i] : col[i];
                            __builtin_amdgcn_wave_barrier();
                        });
                        condest = 1.0 / rows_rcond<NM>(h, col, rd, anorm, lane);
                    }
                }
                if (iter >= maxit || !ok || t == 0.0 || condest > A.cond_h_max) {
                    do_reg = true;                              // opt.cpp:244
                } else {
                    bool stop = err <= sr[4 * S_RTOL];
                    if (A.tol_gamma > 0.0) {
                        const double da1 = row_sum(in ? fabs(x) : 0.0);
                        stop = stop && gamma_ok(A, da1, PPN);
                    }
                    if (stop) {
                        converged = true;                       // opt.cpp:293-306
                    } else {                                    // linesearch.cpp:28-43
                        const double di = in ? -x : 0.0;
                        const double maxf = row_max(in ? fabs(di) / (fabs(al) + 1e-100) : 0.0);
                        vl[64 * V_AOLD] = al;
                        vl[64 * V_DL] = di;
                        sr[4 * S_MAXF] = maxf;
                        sr[4 * S_GD] = row_sum(gv * di);
                        sr[4 * S_FCUR] = fcur;
                        sr[4 * S_FSCALE] = fscale;
                        t = 1.0;
                        if (t * maxf > DBL_EPSILON / 2) {
                            al = al + di;
                            mode = ST_TRIAL;
                        } else {
                            t = 0.0;
                            ++iter; ++total;
                            do_reg = true;
                        }
                    }
                }
            }
            if (do_reg && !PPN && net_fallback(A, reg, warm, iter)) {   // the network's guess failed
                warm = kWarmFellBack;
                if (owner && r == 0) {
                    St{A.st_d, A.st_i, A.cap}.i(St::I_WARM, c) = kWarmFellBack;
                    ++st[R_FALLBACK];
                }
                al = r == 0 ? 2.0 * kSqrtPi * log(0.5 / kSqrtPi) : 0.0;
                iter = 0;
                t = 1.0;
                mode = ST_NEWTON;
            } else if (do_reg) {                                // opt.cpp:246-273
                if (reg < 4) {
                    ++reg;
                    const double rr = kReg[reg];
                    const double uk = r == 0 ? 1.0 : (in ? (A.u[size_t(c) * NM + r] / sr[4 * S_U0]) * (1.0 - rr) : 0.0);
                    vl[64 * V_UL] = uk;
                    sr[4 * S_RTOL] = sqrt(row_sum(uk * uk)) * A.tol;
                    al = r == 0 ? (PPN ? 1.0 - 4.0 * sr[4 * S_DELTA] * kPi : 2.0 * kSqrtPi * log(0.5 / kSqrtPi)) : 0.0;
                    iter = 0;
                    t = 1.0;
                    if (reg == 4) maxit = 10 * maxit;
                    mode = ST_NEWTON;
                } else {                                        // "Max regularization achieved."
                    if (owner && r == 0) {
                        st[R_ERR] |= 1 << MNC_ERR_MAXREG;
                        if (A.outs) { A.outs[c].iter = total; A.outs[c].r = -1.0; A.outs[c].norm_g = err; }
                    }
                    done = true;
                }
            } else if (converged) {
                const double u0 = sr[4 * S_U0];
                double un, an;
                if (PPN) {                                      // no reconstruction; opt.cpp:131-136
                    un = ul * u0;
                    an = al * u0;
                } else {                                        // :298-302, opt.cpp:107-109
                    const double u0p = row_bcast<0>(ul) + row_bcast<0>(gv);
                    un = ((ul + gv) / u0p) * u0;
                    an = r == 0 ? (al - log(u0p) * 2.0 * kSqrtPi) + sr[4 * S_ASCALE] : al;
                }
                if (owner && in) {
                    A.u[size_t(c) * NM + r] = un;
                    A.alpha[size_t(c) * NM + r] = an;
                }
                if (owner && r == 0) {
                    if (A.outs) { A.outs[c].iter = total; A.outs[c].r = kReg[reg]; A.outs[c].norm_g = err; }
                    st[R_MAX_ITER] = max(total, st[R_MAX_ITER]);
                    st[R_SUM] += total;
                    ++st[R_N];
                    ++st[R_HIST + reg];
                }
                done = true;
            }
            if (done) c = -1;
        }
        __builtin_amdgcn_wave_barrier();
    }
    // statistics: the block's counts, one atomic each
    static_assert(kRowCounts == 15, "one thread per count below");
    lane = threadIdx.x & 63;
    if (lane < kRowCounts) {
        const int *n = counts + lane;
        const int x[4] = {n[0], n[kRowCounts], n[2 * kRowCounts], n[3 * kRowCounts]};
        int v = lane == R_MAX_ITER ? max(max(x[0], x[1]), max(x[2], x[3]))
                                   : (lane == R_ERR ? x[0] | x[1] | x[2] | x[3] : x[0] + x[1] + x[2] + x[3]);
        if (lane == R_TITER) {          // less what the listed cells brought with them
            const int *m = counts + R_SUM;
            v += m[0] + m[kRowCounts] + m[2 * kRowCounts] + m[3 * kRowCounts];
        }
        red[wave][lane] = v;
    }
    __syncthreads();
    if (threadIdx.x < 15) {
        const int i = threadIdx.x;
        long long s = 0;
        for (int w = 0; w < kRowWaves; ++w) s = i == 0 ? max(s, (long long)red[w][i]) : (i == 1 ? s | red[w][i] : s + red[w][i]);
        constexpr int word[15] = {0, -1, 1, 2, 8, 3, 4, 5, 6, 7, 13, 14, 16, 10, 11};
        int dst = 0;
#pragma unroll
        for (int k = 0; k < 15; ++k) dst = k == i ? word[k] : dst;
        if (s != 0) {
            if (i == 0) atomicMax((unsigned long long *)&A.stats[0], (unsigned long long)s);
            else if (i == 1) atomicOr(&A.ctl[3], int(s));
            else atomicAdd((unsigned long long *)&A.stats[dst], (unsigned long long)s);
            if (i == 4) atomicAdd((unsigned long long *)&A.stats[15], (unsigned long long)s);
        }
    }
}

constexpr int kRowLdsBytes = 64 * 1024;      // the orbit table in LDS while it and the waves' words fit, else read from L2

template <int N, bool GAUNT, bool PPN, bool WIDE>
void launch_rows_w(const NewtonArgs &a, int blocks, int lin, int lin2, bool fresh, bool few, hipStream_t s) {
    using Dm = RowDims<N, GAUNT, PPN, WIDE>;
    const size_t table = size_t(Dm::NP2 + 1) * a.nop * sizeof(double);
    const size_t own = size_t(kRowWaves) * Dm::LANE_WORDS * sizeof(double);
    const dim3 g(blocks), b(64 * kRowWaves);
    if (table + own <= size_t(kRowLdsBytes) - 512)
        hipLaunchKernelGGL((rows_kernel<N, GAUNT, PPN, WIDE, true>), g, b, table + own, s, a, lin, lin2, int(fresh), int(few));
    else
        hipLaunchKernelGGL((rows_kernel<N, GAUNT, PPN, WIDE, false>), g, b, own, s, a, lin, lin2, int(fresh), int(few));
}

template <int N, bool GAUNT, bool PPN>
void launch_rows_n(const NewtonArgs &a, int lin, int lin2, bool fresh, int num_cu, int tail_blocks, hipStream_t s) {
    // A cell per wave shortens one evaluation (one orbit per lane at Q = 16, not
    // four); four cells per wave share the algebra's issue slots and take a quarter
    // of the waves.  The first wins while every cell has a SIMD to itself.  Kernel us,
    // one cell per wave and four, Q = 16 (M2: 12):
    //   closures          256      1,024     2,048     4,096     8,192
    //   M4 cold          70  91    86 100   119 103   192 116   305 163
    //   M4 near starts   40  47    52  51    76  55   112  66   177  94
    //   M2 near starts   23  28    36  29    59  34    83  44   130  69
    // The four-cell form fills the chip, at two waves per SIMD, from 8,192 cells on; below,
    // some of it idles, and the time is the evaluations' latency.
    // Against the lockstep kernels and a tail of one wave per cell (the whole call,
    // M4, Q = 16): 2,049 closures from near starts 1.01 -> 0.09 ms, 150,001 cold ones
    // with a fifth near the realizability boundary 12.3 -> 2.85; 60 of M2 320 -> 71 us.
    if (fresh) {
        const int waves = 4 * num_cu;                         // one per SIMD
        if (a.ncells <= waves) {
            launch_rows_w<N, GAUNT, PPN, true>(a, (a.ncells + kRowWaves - 1) / kRowWaves, lin, lin2, true, false, s);
        } else {
            const int want = (a.ncells + 4 * kRowWaves - 1) / (4 * kRowWaves);
            launch_rows_w<N, GAUNT, PPN, false>(a, want < 2 * num_cu ? want : 2 * num_cu, lin, lin2, true, false, s);
        }
        return;
    }
    const bool few = a.ncells > tail_blocks * kRowWaves;       // else every list fits one cell per wave
    launch_rows_w<N, GAUNT, PPN, true>(a, tail_blocks, lin, lin2, false, few, s);
    if (few) launch_rows_w<N, GAUNT, PPN, false>(a, tail_blocks, lin, lin2, false, true, s);
}

}  // namespace

bool launch_rows(const NewtonArgs &a, int nm, bool gaunt, int lin, int lin2, bool fresh, int num_cu, int tail_blocks,
                 hipStream_t s) {
#define MNC_ROWS(N)                                                                                          \
    if (nm == orbit_nm(N)) {                                                                                 \
        if (gaunt) {                                                                                         \
            if (a.ppn) launch_rows_n<N, true, true>(a, lin, lin2, fresh, num_cu, tail_blocks, s);            \
            else launch_rows_n<N, true, false>(a, lin, lin2, fresh, num_cu, tail_blocks, s);                 \
        } else {                                                                                             \
            if (a.ppn) launch_rows_n<N, false, true>(a, lin, lin2, fresh, num_cu, tail_blocks, s);           \
            else launch_rows_n<N, false, false>(a, lin, lin2, fresh, num_cu, tail_blocks, s);                \
        }                                                                                                    \
        return true;                                                                                         \
    }
    MNC_ROWS(0)
    MNC_ROWS(1)
    MNC_ROWS(2)
    MNC_ROWS(3)
    MNC_ROWS(4)
#undef MNC_ROWS
    return false;
}

}  // namespace mnc
