// mnc_grid.hip -- ansatz, kinetic flux, Euler/Heun stage and ghost fill of the
// Mn solver on gfx950 (src/momopt/momopt_update.cpp:38-202,283-382 and
// src/momopt/momopt_boundaries.cpp:190-223).
//
// Data layout in HBM: grid arrays are the reference's I3D layout
// [(i*(ny+4)+j)][k] (x-major, 2 ghost cells per side); the ansatz is stored
// [q][cell] so that, for one quadrature direction, neighbouring threads (cells)
// read neighbouring words.
#include <algorithm>
#include <type_traits>

#include "mnc_internal.h"
#include "mnc_orbit.h"

namespace mnc {
namespace {

// The left edge x0 + k h of a cell for the lattice source test |x| < 0.5
// (momopt_update.cpp:328-334), rounded as a product and a sum, as the
// reference's x86-64 build without FMA evaluates it: on grids whose edges
// fall on +-0.5 exactly (280 cells on [-3.5, 3.5]: h = 0.025) a contracted
// fma lands inside and adds a row and a column of source cells.
// (__dadd_rn / __dmul_rn alone do not stop the contraction: the pragma does.)
__device__ __forceinline__ double edge_coord(double x0, int k, double h) {
#pragma clang fp contract(off)
    return x0 + double(k) * h;
}

constexpr int kBlock = 256;

// momopt_update.cpp:77-90 (SIGN/MIN/MAX of utils.h:28-30)
__device__ __forceinline__ double sgn1(double x) { return (x >= 0.0) ? 1.0 : -1.0; }
__device__ __forceinline__ double minmod(double x, double y) {
    const double a = fabs(x), b = y * sgn1(x);
    const double mn = (a < b) ? a : b;
    return sgn1(x) * ((0.0 > mn) ? 0.0 : mn);
}
__device__ __forceinline__ double slopefit(double l, double c, double r, double theta) {
    return minmod(theta * (r - c), minmod(0.5 * (r - l), theta * (c - l)));
}

// The Euler stage of interior cell (i, j) = c with flux F (:316-336 / :344-364),
// the lattice source (:328-334) and, on the second stage, the Heun average
// (:368-377); stage 0 stores the flux only.
template <int NM>
__device__ __forceinline__ void euler_epilogue(const GridArgs &g, int i, int j, size_t c, const double (&F)[NM],
                                               int stage, double dt) {
    if (stage == 0) {
#pragma unroll
        for (int k = 0; k < NM; ++k) g.flux[c * NM + k] = F[k];
        return;
    }
    double *u = g.moments + c * NM;
    const double st = g.sigma_t[c], ss = g.sigma_s[c];
    double v[NM];
    v[0] = u[0] * (1.0 + dt * ss - dt * st) - dt * F[0];
#pragma unroll
    for (int k = 1; k < NM; ++k) v[k] = u[k] * (1.0 - dt * st) - dt * F[k];
    if (g.init_cond == 1) {
        const double x_i = edge_coord(g.init_x, i - 2, g.dx);
        const double y_j = edge_coord(g.init_y, j - 2, g.dy);
        if (fabs(x_i) < 0.5 && fabs(y_j) < 0.5) v[0] = v[0] + dt * 2.0 * sqrt(M_PI);
    }
    if (stage == 2) {
        const double *uo = g.moments_old + c * NM;
#pragma unroll
        for (int k = 0; k < NM; ++k) v[k] = 0.5 * (v[k] + uo[k]);
    }
#pragma unroll
    for (int k = 0; k < NM; ++k) u[k] = v[k];
}

// The ansatz at kinetic = alpha.m_q (computeAnsatz, :38-58): exp for Mn; for
// PPn kinetic/2 + sqrt(kinetic^2 + 4 delta)/2, written for kinetic <= 0 in
// the form without cancellation.
__device__ __forceinline__ double ansatz_value(const GridArgs &g, double kinetic) {
    if (g.ppn) {
        if (kinetic > 0) return 0.5 * kinetic + 0.5 * sqrt(kinetic * kinetic + 4 * g.delta);
        return -g.delta / (0.5 * kinetic - 0.5 * sqrt(kinetic * kinetic + 4 * g.delta));
    }
    return exp(kinetic);
}

// E[q][cell] = ansatz(alpha_cell . m_q) for q in [q0, q0+nqc)  (computeAnsatz, :38-58)
template <int NM>
__global__ __launch_bounds__(kBlock) void ansatz_kernel(GridArgs g, int q0, int nqc) {
    const int ncell = g.NX * g.NY;
    const int c = blockIdx.x * kBlock + threadIdx.x;
    if (c >= ncell) return;
    double a[NM];
#pragma unroll
    for (int k = 0; k < NM; ++k) a[k] = g.alpha[size_t(c) * NM + k];
    for (int qq = 0; qq < nqc; ++qq) {
        const double *row = g.p + size_t(q0 + qq) * g.np2;
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < NM; ++k) s = fma(a[k], row[k], s);
        g.ansatz[size_t(qq) * ncell + c] = ansatz_value(g, s);
    }
}

// Interior flux (solveFlux :128-196) accumulated over q in [q0, q0+nqc) in
// ascending q, then (last chunk) the Euler stage (:316-336 / :344-364) and, on
// the second stage, the Heun average (:368-377).
template <int NM>
__global__ __launch_bounds__(kBlock) void flux_euler_kernel(GridArgs g, int q0, int nqc, int stage, double dt,
                                                             int first_chunk, int last_chunk) {
    const int idx = blockIdx.x * kBlock + threadIdx.x;
    if (idx >= g.nx * g.ny) return;
    const int i = 2 + idx / g.ny;
    const int j = 2 + idx % g.ny;
    const int NY = g.NY;
    const int ncell = g.NX * g.NY;
    const size_t c = size_t(i) * NY + j;
    double F[NM];
    if (first_chunk) {
#pragma unroll
        for (int k = 0; k < NM; ++k) F[k] = 0.0;
    } else {
#pragma unroll
        for (int k = 0; k < NM; ++k) F[k] = g.flux[c * NM + k];
    }
    const double theta = g.theta, dx = g.dx, dy = g.dy;
    for (int qq = 0; qq < nqc; ++qq) {
        const int q = q0 + qq;
        const double *E = g.ansatz + size_t(qq) * ncell;
        const double xi = g.xi[q], eta = g.eta[q], w = g.w[q];
        double f1 = 0.0, f2 = 0.0, f3 = 0.0, f4 = 0.0;
        if (xi > 0) {
            const double k1 = E[(i - 2) * NY + j], k2 = E[(i - 1) * NY + j];
            const double k3 = E[i * NY + j], k4 = E[(i + 1) * NY + j];
            f1 = k3 + 0.5 * slopefit(k2, k3, k4, theta) - k2 - 0.5 * slopefit(k1, k2, k3, theta);
            f1 = f1 * xi * w;
        }
        if (xi < 0) {
            const double k1 = E[(i - 1) * NY + j], k2 = E[i * NY + j];
            const double k3 = E[(i + 1) * NY + j], k4 = E[(i + 2) * NY + j];
            f2 = k3 - 0.5 * slopefit(k2, k3, k4, theta) - k2 + 0.5 * slopefit(k1, k2, k3, theta);
            f2 = f2 * xi * w;
        }
        if (eta > 0) {
            const double k1 = E[i * NY + (j - 2)], k2 = E[i * NY + (j - 1)];
            const double k3 = E[i * NY + j], k4 = E[i * NY + (j + 1)];
            f3 = k3 + 0.5 * slopefit(k2, k3, k4, theta) - k2 - 0.5 * slopefit(k1, k2, k3, theta);
            f3 = f3 * eta * w;
        }
        if (eta < 0) {
            const double k1 = E[i * NY + (j - 1)], k2 = E[i * NY + j];
            const double k3 = E[i * NY + (j + 1)], k4 = E[i * NY + (j + 2)];
            f4 = k3 - 0.5 * slopefit(k2, k3, k4, theta) - k2 + 0.5 * slopefit(k1, k2, k3, theta);
            f4 = f4 * eta * w;
        }
        const double comb = (f1 + f2) / dx + (f3 + f4) / dy;
        const double *row = g.p + size_t(q) * g.np2;
#pragma unroll
        for (int k = 0; k < NM; ++k) F[k] = fma(row[k], comb, F[k]);
    }
    if (!last_chunk || stage == 0) {
#pragma unroll
        for (int k = 0; k < NM; ++k) g.flux[c * NM + k] = F[k];
        return;
    }
    double *u = g.moments + c * NM;
    const double st = g.sigma_t[c], ss = g.sigma_s[c];
    double v[NM];
    v[0] = u[0] * (1.0 + dt * ss - dt * st) - dt * F[0];
#pragma unroll
    for (int k = 1; k < NM; ++k) v[k] = u[k] * (1.0 - dt * st) - dt * F[k];
    if (g.init_cond == 1) {                                   // lattice source (:328-334)
        const double x_i = edge_coord(g.init_x, i - 2, dx);
        const double y_j = edge_coord(g.init_y, j - 2, dy);
        if (fabs(x_i) < 0.5 && fabs(y_j) < 0.5) v[0] = v[0] + dt * 2.0 * sqrt(M_PI);
    }
    if (stage == 2) {
        const double *uo = g.moments_old + c * NM;
#pragma unroll
        for (int k = 0; k < NM; ++k) v[k] = 0.5 * (v[k] + uo[k]);
    }
#pragma unroll
    for (int k = 0; k < NM; ++k) u[k] = v[k];
}

// The ansatz fused into the flux: a block owns a TX x TY tile of interior cells,
// keeps alpha of the tile and its 2-cell halo in LDS, and for each chunk of QC
// directions evaluates the ansatz E of the halo'd tile into LDS (the halo
// is evaluated by both neighbouring tiles) before the stencil reads it.  E never
// goes to HBM.  The arithmetic of every cell is that of ansatz_kernel +
// flux_euler_kernel (same summation order over k and q), so the results are
// identical.
template <int NM, int TX, int TY, int QC>
__global__ __launch_bounds__(TX * TY) void flux_fused_kernel(GridArgs g, int stage, double dt) {
    constexpr int HX = TX + 4, HY = TY + 4, NH = HX * HY, NT = TX * TY;
    __shared__ double al_s[NH][NM];
    __shared__ double E_s[QC][NH];
    const int tid = threadIdx.x;
    const int tx0 = blockIdx.x * TX, ty0 = blockIdx.y * TY;   // halo cell (hi, hj) is grid cell (tx0+hi, ty0+hj)
    const int NX = g.NX, NY = g.NY;
    for (int idx = tid; idx < NH * NM; idx += NT) {
        const int h = idx / NM, k = idx % NM;
        const int gi = tx0 + h / HY, gj = ty0 + h % HY;
        al_s[h][k] = (gi < NX && gj < NY) ? g.alpha[(size_t(gi) * NY + gj) * NM + k] : 0.0;
    }
    const int li = tid / TY, lj = tid % TY;
    const int i = 2 + tx0 + li, j = 2 + ty0 + lj;
    const bool active = (tx0 + li < g.nx) && (ty0 + lj < g.ny);
    const int hc = (li + 2) * HY + (lj + 2);                  // this cell's halo index
    const double theta = g.theta, dx = g.dx, dy = g.dy;
    double F[NM];
#pragma unroll
    for (int k = 0; k < NM; ++k) F[k] = 0.0;
    for (int q0 = 0; q0 < g.nq; q0 += QC) {
        const int nqc = min(QC, g.nq - q0);
        __syncthreads();
        for (int qq = 0; qq < nqc; ++qq) {
            const double *row = g.p + size_t(q0 + qq) * g.np2;
            for (int h = tid; h < NH; h += NT) {
                double sa = 0.0;
#pragma unroll
                for (int k = 0; k < NM; ++k) sa = fma(al_s[h][k], row[k], sa);
                E_s[qq][h] = ansatz_value(g, sa);
            }
        }
        __syncthreads();
        if (!active) continue;
        for (int qq = 0; qq < nqc; ++qq) {
            const int q = q0 + qq;
            const double *E = E_s[qq];
            const double xi = g.xi[q], eta = g.eta[q], w = g.w[q];
            double f1 = 0.0, f2 = 0.0, f3 = 0.0, f4 = 0.0;
            if (xi > 0) {
                const double k1 = E[hc - 2 * HY], k2 = E[hc - HY], k3 = E[hc], k4 = E[hc + HY];
                f1 = k3 + 0.5 * slopefit(k2, k3, k4, theta) - k2 - 0.5 * slopefit(k1, k2, k3, theta);
                f1 = f1 * xi * w;
            }
            if (xi < 0) {
                const double k1 = E[hc - HY], k2 = E[hc], k3 = E[hc + HY], k4 = E[hc + 2 * HY];
                f2 = k3 - 0.5 * slopefit(k2, k3, k4, theta) - k2 + 0.5 * slopefit(k1, k2, k3, theta);
                f2 = f2 * xi * w;
            }
            if (eta > 0) {
                const double k1 = E[hc - 2], k2 = E[hc - 1], k3 = E[hc], k4 = E[hc + 1];
                f3 = k3 + 0.5 * slopefit(k2, k3, k4, theta) - k2 - 0.5 * slopefit(k1, k2, k3, theta);
                f3 = f3 * eta * w;
            }
            if (eta < 0) {
                const double k1 = E[hc - 1], k2 = E[hc], k3 = E[hc + 1], k4 = E[hc + 2];
                f4 = k3 - 0.5 * slopefit(k2, k3, k4, theta) - k2 + 0.5 * slopefit(k1, k2, k3, theta);
                f4 = f4 * eta * w;
            }
            const double comb = (f1 + f2) / dx + (f3 + f4) / dy;
            const double *row = g.p + size_t(q) * g.np2;
#pragma unroll
            for (int k = 0; k < NM; ++k) F[k] = fma(row[k], comb, F[k]);
        }
    }
    if (!active) return;
    const size_t c = size_t(i) * NY + j;
    if (stage == 0) {
#pragma unroll
        for (int k = 0; k < NM; ++k) g.flux[c * NM + k] = F[k];
        return;
    }
    double *u = g.moments + c * NM;
    const double st = g.sigma_t[c], ss = g.sigma_s[c];
    double v[NM];
    v[0] = u[0] * (1.0 + dt * ss - dt * st) - dt * F[0];
#pragma unroll
    for (int k = 1; k < NM; ++k) v[k] = u[k] * (1.0 - dt * st) - dt * F[k];
    if (g.init_cond == 1) {                                   // lattice source (:328-334)
        const double x_i = edge_coord(g.init_x, i - 2, dx);
        const double y_j = edge_coord(g.init_y, j - 2, dy);
        if (fabs(x_i) < 0.5 && fabs(y_j) < 0.5) v[0] = v[0] + dt * 2.0 * sqrt(M_PI);
    }
    if (stage == 2) {
        const double *uo = g.moments_old + c * NM;
#pragma unroll
        for (int k = 0; k < NM; ++k) v[k] = 0.5 * (v[k] + uo[k]);
    }
#pragma unroll
    for (int k = 0; k < NM; ++k) u[k] = v[k];
}

// duplicateBoundaries (momopt_boundaries.cpp:190-223): x strips, then y strips.
__global__ void ghost_x_kernel(GridArgs g) {
    const int idx = blockIdx.x * kBlock + threadIdx.x;   // over 2 * ny * nm
    const int total = 2 * g.ny * g.nm;
    if (idx >= total) return;
    const int k = idx % g.nm;
    const int j = 2 + (idx / g.nm) % g.ny;
    const int i = idx / (g.nm * g.ny);
    const int x0 = 0, x1 = 2, x2 = 2 + g.nx - 2, x3 = 2 + g.nx;
    const int NY = g.NY, nm = g.nm;
    g.moments[(size_t(x0 + i) * NY + j) * nm + k] = g.moments[(size_t(x2 + i) * NY + j) * nm + k];
    g.moments[(size_t(x3 + i) * NY + j) * nm + k] = g.moments[(size_t(x1 + i) * NY + j) * nm + k];
}

__global__ void ghost_y_kernel(GridArgs g) {
    const int idx = blockIdx.x * kBlock + threadIdx.x;   // over nx * 2 * nm
    const int total = g.nx * 2 * g.nm;
    if (idx >= total) return;
    const int k = idx % g.nm;
    const int jj = (idx / g.nm) % 2;
    const int i = 2 + idx / (g.nm * 2);
    const int y0 = 0, y1 = 2, y2 = 2 + g.ny - 2, y3 = 2 + g.ny;
    const int NY = g.NY, nm = g.nm;
    g.moments[(size_t(i) * NY + y0 + jj) * nm + k] = g.moments[(size_t(i) * NY + y2 + jj) * nm + k];
    g.moments[(size_t(i) * NY + y3 + jj) * nm + k] = g.moments[(size_t(i) * NY + y1 + jj) * nm + k];
}

// minmod(theta (r - c), (r - l) / 2, theta (c - l)): 0 unless all three share
// their sign, else the smallest magnitude with it (slopefit's values).
__device__ __forceinline__ double slope3(double l, double c, double r, double theta) {
    const double a = theta * (r - c), b = theta * (c - l), m = 0.5 * (r - l);
    const double v = fmin(fmin(fabs(a), fabs(b)), fabs(m));
    const int s = __double2hiint(m);
    return ((__double2hiint(a) ^ s) | (__double2hiint(b) ^ s)) < 0 ? 0.0 : copysign(v, m);
}

// Difference of the face values around c for the upwind side `up` (+1: the wind
// comes from below).
template <int UP>
__device__ __forceinline__ double face_diff(double m2, double m1, double c, double p1, double p2, double theta) {
    if constexpr (UP > 0) return c + 0.5 * slope3(m1, c, p1, theta) - m1 - 0.5 * slope3(m2, m1, c, theta);
    else return p1 - 0.5 * slope3(c, p1, p2, theta) - c + 0.5 * slope3(m1, c, p1, theta);
}

template <class T>
__device__ __forceinline__ void each_class(T &&f) {
    f(std::integral_constant<int, 0>{});
    f(std::integral_constant<int, 1>{});
    f(std::integral_constant<int, 2>{});
    f(std::integral_constant<int, 3>{});
}

template <int NM> constexpr int order_of_nm() {
    int N = 0;
    while (orbit_nm(N) < NM) ++N;
    return N;
}
template <int NM> struct Classes {
    unsigned char of[NM];
    constexpr Classes() : of{} {
        for (int k = 0; k < NM; ++k) of[k] = (unsigned char)orbit_class(k);
    }
};

// The fused ansatz + flux with the quadrature's orbits (mnc_orbit.h) split into
// gridDim.z groups: block (tile, z) sums the flux of its TX x TY cells over group
// z's orbits into fpart[z] (interior cells, [cell][k]), and flux_sum_kernel adds
// the groups in order and applies the Euler stage.  Per chunk of OC orbits the
// ansatz at their four images goes to LDS for the tile and its halo of two cells
// (evaluated by both neighbouring tiles; alpha of a thread's halo cells stays in
// registers), then each thread takes its cell's stencil.  Bound by FP64 issue, some
// 500 instructions per orbit and cell: the four images share one pass over the
// moments before the ansatz and one after the stencil, their upwind sides are
// known when compiled, and a slope is thirteen instructions.  Direction by
// direction (two passes of n FMAs, branches on the signs, slopes of selects) M4,
// Q = 16 took 190 us a stage at 280^2 and 63 at 133 x 101; now 133 and 45.
template <int NM, int TX, int TY, int OC>
__global__ __launch_bounds__(TX * TY) void flux_split_kernel(GridArgs g) {
    static_assert(TX == kSplitTile && TY == kSplitTile, "the tile flags' geometry");
    if (g.tile_mode != 0) {   // this launch's share of the tiles (uniform over the block)
        const bool flagged = g.tile_flag[blockIdx.x * gridDim.y + blockIdx.y] != 0;
        if (flagged != (g.tile_mode == 2)) return;
    }
    constexpr Classes<NM> cls{};
    constexpr int HX = TX + 4, HY = TY + 4, NH = HX * HY, NT = TX * TY;
    constexpr int HPT = (NH + NT - 1) / NT;                  // halo cells evaluated per thread
    __shared__ double E_s[4 * OC][NH];
    const int tid = threadIdx.x;
    const int tx0 = blockIdx.x * TX, ty0 = blockIdx.y * TY;
    const int NX = g.NX, NY = g.NY;
    double al[HPT][NM];
#pragma unroll
    for (int hh = 0; hh < HPT; ++hh) {
        const int h = tid + hh * NT;
        const int gi = tx0 + h / HY, gj = ty0 + h % HY;
        const bool in = h < NH && gi < NX && gj < NY;
#pragma unroll
        for (int k = 0; k < NM; ++k) al[hh][k] = in ? g.alpha[(size_t(gi) * NY + gj) * NM + k] : 0.0;
    }
    const int li = tid / TY, lj = tid % TY;
    const int i = 2 + tx0 + li, j = 2 + ty0 + lj;
    const bool active = (tx0 + li < g.nx) && (ty0 + lj < g.ny);
    const int hc = (li + 2) * HY + (lj + 2);
    const double theta = g.theta, rdx = 1.0 / g.dx, rdy = 1.0 / g.dy;
    const int half = g.half, no = half * half;
    const int per = (no + gridDim.z - 1) / gridDim.z;
    const int oa = blockIdx.z * per, ob = min(no, oa + per);
    auto node = [&](int o) { return 4 * half * (o / half) + o % half; };   // the orbit's node with xi, eta > 0
    double F[NM];
#pragma unroll
    for (int k = 0; k < NM; ++k) F[k] = 0.0;
    for (int o0 = oa; o0 < ob; o0 += OC) {
        const int noc = min(OC, ob - o0);
        __syncthreads();
        for (int oo = 0; oo < noc; ++oo) {
            const double *row = g.p + size_t(node(o0 + oo)) * g.np2;
#pragma unroll
            for (int hh = 0; hh < HPT; ++hh) {
                const int h = tid + hh * NT;
                if (h < NH) {
                    double z[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
                    for (int k = 0; k < NM; ++k) z[cls.of[k]] = fma(al[hh][k], row[k], z[cls.of[k]]);
                    const double ep = z[0] + z[1], em = z[0] - z[1], op = z[2] + z[3], om = z[2] - z[3];
                    E_s[4 * oo][h] = ansatz_value(g, ep + op);
                    E_s[4 * oo + 1][h] = ansatz_value(g, em + om);         // -xi: classes 1 and 3 change sign
                    E_s[4 * oo + 2][h] = ansatz_value(g, ep - op);         // -eta: classes 2 and 3
                    E_s[4 * oo + 3][h] = ansatz_value(g, em - om);         // both: classes 1 and 2
                }
            }
        }
        __syncthreads();
        if (!active) continue;
        for (int oo = 0; oo < noc; ++oo) {
            const int q = node(o0 + oo);
            const double fx = g.xi[q] * g.w[q] * rdx, fy = g.eta[q] * g.w[q] * rdy;
            double comb[4];
            each_class([&](auto img) {
                constexpr int I = decltype(img)::value, UX = I & 1 ? -1 : 1, UY = I & 2 ? -1 : 1;
                const double *e = &E_s[4 * oo + I][hc];
                const double c = e[0], xm1 = *(e - HY), xp1 = e[HY], ym1 = *(e - 1), yp1 = e[1];
                const double xo = UX > 0 ? *(e - 2 * HY) : e[2 * HY], yo = UY > 0 ? *(e - 2) : e[2];
                comb[I] = UX * fx * face_diff<UX>(xo, xm1, c, xp1, xo, theta) + UY * fy * face_diff<UY>(yo, ym1, c, yp1, yo, theta);
            });
            const double ep = comb[0] + comb[1], em = comb[0] - comb[1], op = comb[2] + comb[3], om = comb[2] - comb[3];
            const double C[4] = {ep + op, em + om, ep - op, em - om};
            const double *row = g.p + size_t(q) * g.np2;
#pragma unroll
            for (int k = 0; k < NM; ++k) F[k] = fma(row[k], C[cls.of[k]], F[k]);
        }
    }
    if (!active) return;
    double *o = g.fpart + (size_t(blockIdx.z) * g.nx * g.ny + size_t(i - 2) * g.ny + (j - 2)) * NM;
#pragma unroll
    for (int k = 0; k < NM; ++k) o[k] = F[k];
}

// F = fpart[0] + fpart[1] + ... (in group order), then the Euler stage.
template <int NM>
__global__ __launch_bounds__(kBlock) void flux_sum_kernel(GridArgs g, int groups, int stage, double dt) {
    const int idx = blockIdx.x * kBlock + threadIdx.x;
    if (idx >= g.nx * g.ny) return;
    const int i = 2 + idx / g.ny, j = 2 + idx % g.ny;
    if (g.tile_mode != 0) {
        const int tiles_y = (g.ny + kSplitTile - 1) / kSplitTile;
        const bool flagged = g.tile_flag[((i - 2) / kSplitTile) * tiles_y + (j - 2) / kSplitTile] != 0;
        if (flagged != (g.tile_mode == 2)) return;
    }
    double F[NM];
#pragma unroll
    for (int k = 0; k < NM; ++k) F[k] = g.fpart[size_t(idx) * NM + k];
    for (int z = 1; z < groups; ++z) {
        const double *p = g.fpart + (size_t(z) * g.nx * g.ny + idx) * NM;
#pragma unroll
        for (int k = 0; k < NM; ++k) F[k] += p[k];
    }
    euler_epilogue<NM>(g, i, j, size_t(i) * g.NY + j, F, stage, dt);
}

template <int NM>
void launch_fused_t(const GridArgs &g, int tile, int stage, double dt, hipStream_t s) {
    if constexpr (NM <= 15) {   // alpha of two halo cells per thread in registers
        if (tile == 3) {
            const dim3 grid((g.nx + 15) / 16, (g.ny + 15) / 16, g.groups);
            hipLaunchKernelGGL((flux_split_kernel<NM, 16, 16, 2>), grid, dim3(256), 0, s, g);
            hipLaunchKernelGGL((flux_sum_kernel<NM>), dim3((g.nx * g.ny + kBlock - 1) / kBlock), dim3(kBlock), 0, s,
                               g, g.groups, stage, dt);
            return;
        }
    }
    if constexpr (NM <= 15) {   // alpha of a 20 x 20 halo'd tile fits LDS up to n = 15
        if (tile == 2) {
            hipLaunchKernelGGL((flux_fused_kernel<NM, 16, 16, 8>), dim3((g.nx + 15) / 16, (g.ny + 15) / 16), dim3(256),
                               0, s, g, stage, dt);
            return;
        }
    }
    hipLaunchKernelGGL((flux_fused_kernel<NM, 8, 8, 8>), dim3((g.nx + 7) / 8, (g.ny + 7) / 8), dim3(64), 0, s, g,
                       stage, dt);
}

// ---- flux of the orders 5 to 8 through HBM, on the matrix cores ---------------
//
// The ansatz at the four images of an orbit (mnc_orbit.h) needs one pass over the
// moments: z = sum of four class sums with signs; and the moments of the four
// fluxes one pass back: F_k = sum over orbits of m_k C[class of k], C the signed
// sums of the images' fluxes.  Both passes are products on the matrix cores,
// sixteen cells a wave.
//
// A lane per cell and one direction at a time these were 965 us (ansatz) and
// 1,709 us (flux) at 96 x 96 M8 cells and 1,024 directions, on 40 blocks and a
// serial walk over all directions; the products are a quarter of the FMAs, and
// the two take 31 and 75 us.

typedef double gf64x4 __attribute__((ext_vector_type(4)));

template <int N>
struct FluxShape {
    static constexpr int kz(int c) { return (orbit_class_size(N, c) + 3) / 4; }
    static constexpr int k0(int c) { return c == 0 ? 0 : k0(c - 1) + kz(c - 1); }
    static constexpr int KZ = k0(4);
};
// E[4 orbit + image][cell] of the orbit tiles T0 .. T0 + ntc - 1.  A wave takes 16
// cells and every gridDim.y-th tile.  Bound by the exponentials and the store (82 MB at 96^2).
template <int N>
__global__ __launch_bounds__(256) void ansatz_orbit_kernel(GridArgs g, int T0, int ntc) {
    using F = FluxShape<N>;
    constexpr int NM = orbit_nm(N);
    const int ncell = g.NX * g.NY;
    const int lane = threadIdx.x & 63, q = lane >> 4;
    const int cell = (blockIdx.x * 4 + (threadIdx.x >> 6)) * 16 + (lane & 15);
    const int src = min(cell, ncell - 1);
    double al[F::KZ];
    each_class([&](auto C) {
        constexpr int c = decltype(C)::value, n = F::kz(c), at = F::k0(c);
#pragma unroll
        for (int kk = 0; kk < n; ++kk) {
            const int k = g.oidx[c * 16 + 4 * kk + q];
            al[at + kk] = k >= 0 ? g.alpha[size_t(src) * NM + k] : 0.0;
        }
    });
    for (int T = blockIdx.y; T < ntc; T += gridDim.y) {
        const double *zt = g.oz + size_t(T0 + T) * F::KZ * 64 + lane;
        gf64x4 z[4];
        each_class([&](auto C) {
            constexpr int c = decltype(C)::value, n = F::kz(c), at = F::k0(c);
            z[c] = gf64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int kk = 0; kk < n; ++kk)
                z[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(zt[(at + kk) * 64], al[at + kk], z[c], 0, 0, 0);
        });
        if (cell >= ncell) continue;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            double *E = g.ansatz + size_t(64 * T + 4 * mfma_f64_row(r, q)) * ncell + cell;
            const double ep = z[0][r] + z[1][r], em = z[0][r] - z[1][r], op = z[2][r] + z[3][r], om = z[2][r] - z[3][r];
            E[0] = ansatz_value(g, ep + op);
            E[size_t(ncell)] = ansatz_value(g, em + om);             // -xi: classes 1 and 3 change sign
            E[2 * size_t(ncell)] = ansatz_value(g, ep - op);         // -eta: classes 2 and 3
            E[3 * size_t(ncell)] = ansatz_value(g, em - om);         // both: classes 1 and 2
        }
    }
}

constexpr int kFluxWaves = 8;

// Flux of sixteen interior cells a block, then the Euler stage; the block's waves
// share the steps of four orbits (lane: cell lane % 16, orbit lane / 16), so that
// 96^2 cells are 4,608 waves.  Bound by the L1/L2 reads of the stencil (28 words a
// cell and orbit; XCD b % 8 owns a contiguous range of cells so that the x
// neighbours' rows stay in its L2).
template <int N>
__global__ __launch_bounds__(64 * kFluxWaves) void flux_orbit_kernel(GridArgs g, int T0, int ntc, int stage, double dt,
                                                                     int first_chunk, int last_chunk) {
    constexpr int NM = orbit_nm(N);
    __shared__ double red[4][16][64];
    const int cells = g.nx * g.ny, tiles = (cells + 15) / 16, per = (tiles + 7) / 8;
    const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= per || tile >= tiles) return;           // uniform over the block
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, q = lane >> 4;
    const size_t ncell = size_t(g.NX) * g.NY, NY = g.NY;
    const int idx = min(tile * 16 + (lane & 15), cells - 1);
    const size_t at = size_t(2 + idx / g.ny) * NY + 2 + idx % g.ny;
    const double theta = g.theta, rdx = 1.0 / g.dx, rdy = 1.0 / g.dy;
    gf64x4 acc[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[c] = gf64x4{0.0, 0.0, 0.0, 0.0};
    for (int s = wv; s < 4 * ntc; s += kFluxWaves) {
        const int o = 4 * s + q;
        const double *d = g.odir + size_t(16 * T0 + o) * 4;
        const double fx = d[0] * d[2] * rdx, fy = d[1] * d[2] * rdy;
        const double *E = g.ansatz + size_t(4 * o) * ncell + at;
        const double *pt = g.op + size_t(4 * T0 + s) * 256 + lane;
        double comb[4];
        auto image = [&](auto img) {
            constexpr int I = decltype(img)::value;
            constexpr int UX = I & 1 ? -1 : 1, UY = I & 2 ? -1 : 1;
            const double *e = E + size_t(I) * ncell;
            const double c = e[0], xm1 = *(e - NY), xp1 = e[NY], ym1 = *(e - 1), yp1 = e[1];
            const double xo = UX > 0 ? *(e - 2 * NY) : e[2 * NY], yo = UY > 0 ? *(e - 2) : e[2];
            comb[I] = UX * fx * face_diff<UX>(xo, xm1, c, xp1, xo, theta) + UY * fy * face_diff<UY>(yo, ym1, c, yp1, yo, theta);
        };
        each_class(image);
        const double ep = comb[0] + comb[1], em = comb[0] - comb[1], op = comb[2] + comb[3], om = comb[2] - comb[3];
        const double C[4] = {ep + op, em + om, ep - op, em - om};
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(C[c], pt[c * 64], acc[c], 0, 0, 0);
    }
    // the waves' sums: 4 .. 7 onto 0 .. 3, then wave c takes class c of those four
    auto put = [&](int v) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) red[v][4 * c + r][lane] = acc[c][r];
    };
    if (wv >= 4) put(wv - 4);
    __syncthreads();
    if (wv < 4) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[c][r] += red[wv][4 * c + r][lane];
        put(wv);
    }
    __syncthreads();
    if (wv >= 4) return;
    // element r of lane l: cell mfma_f64_row(r, l / 16), moment l % 16 of the class
    const int k = g.oidx[wv * 16 + (lane & 15)];
    if (k < 0) return;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int id = tile * 16 + mfma_f64_row(r, q);
        if (id >= cells) continue;
        const int i = 2 + id / g.ny, j = 2 + id % g.ny;
        const size_t cc = size_t(i) * NY + j, o = cc * NM + k;
        double Fk = (red[0][4 * wv + r][lane] + red[1][4 * wv + r][lane]) + (red[2][4 * wv + r][lane] + red[3][4 * wv + r][lane]);
        if (!first_chunk) Fk += g.flux[o];
        if (!last_chunk || stage == 0) {
            g.flux[o] = Fk;
            continue;
        }
        // the Euler stage of euler_epilogue, one moment a lane
        const double st = g.sigma_t[cc], u = g.moments[o];
        double v;
        if (k == 0) {
            v = u * (1.0 + dt * g.sigma_s[cc] - dt * st) - dt * Fk;
            if (g.init_cond == 1 && fabs(edge_coord(g.init_x, i - 2, g.dx)) < 0.5 && fabs(edge_coord(g.init_y, j - 2, g.dy)) < 0.5)
                v = v + dt * 2.0 * sqrt(M_PI);
        } else {
            v = u * (1.0 - dt * st) - dt * Fk;
        }
        if (stage == 2) v = 0.5 * (v + g.moments_old[o]);
        g.moments[o] = v;
    }
}

template <int NM>
void launch_ansatz_orbit(const GridArgs &g, int T0, int ntc, hipStream_t s) {
    const int bx = (g.NX * g.NY + 63) / 64;
    const int by = std::min(ntc, std::max(1, 1024 / bx));      // about four waves per SIMD
    hipLaunchKernelGGL(ansatz_orbit_kernel<order_of_nm<NM>()>, dim3(bx, by), dim3(256), 0, s, g, T0, ntc);
}

template <int NM>
void launch_flux_orbit(const GridArgs &g, int T0, int ntc, int stage, double dt, bool fc, bool lc, hipStream_t s) {
    const int tiles = (g.nx * g.ny + 15) / 16;
    hipLaunchKernelGGL(flux_orbit_kernel<order_of_nm<NM>()>, dim3(8 * ((tiles + 7) / 8)), dim3(64 * kFluxWaves), 0, s, g,
                       T0, ntc, stage, dt, int(fc), int(lc));
}

template <int NM>
void launch_flux_t(const GridArgs &g, int q0, int nqc, int stage, double dt, bool fc, bool lc, hipStream_t s) {
    if constexpr (NM > 15) {
        launch_flux_orbit<NM>(g, q0 / 64, nqc / 64, stage, dt, fc, lc, s);
    } else {
        const int n = g.nx * g.ny;
        hipLaunchKernelGGL(flux_euler_kernel<NM>, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, g, q0, nqc,
                           stage, dt, int(fc), int(lc));
    }
}

template <int NM>
void launch_ansatz_t(const GridArgs &g, int q0, int nqc, hipStream_t s) {
    if constexpr (NM > 15) {
        launch_ansatz_orbit<NM>(g, q0 / 64, nqc / 64, s);
    } else {
        const int n = g.NX * g.NY;
        hipLaunchKernelGGL(ansatz_kernel<NM>, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, s, g, q0, nqc);
    }
}

__global__ void tile_flag_clear_kernel(int *flags, int n) {
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) flags[t] = 0;
}

// One thread per list entry: the tiles whose stencil region [16 t, 16 t + 20)
// (grid coordinates, ghosts included) holds the entry's cell.
__global__ void tile_flag_mark_kernel(const int *list0, const int *cnt0, const int *list1, const int *cnt1, int ncells,
                                      int NY, int tiles_x, int tiles_y, int *flags) {
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= ncells) return;
    const int n0 = *cnt0, n1 = *cnt1;
    int c = -1;
    if (s < n0) c = list0[s];
    else if (s - n0 < n1) c = list1[s - n0];
    if (c < 0) return;
    const int ci = c / NY, cj = c % NY;
    constexpr int T = kSplitTile, R = kSplitTile + 4;
    const int tx0 = ci >= R ? (ci - R + T) / T : 0, tx1 = min(tiles_x - 1, ci / T);
    const int ty0 = cj >= R ? (cj - R + T) / T : 0, ty1 = min(tiles_y - 1, cj / T);
    for (int tx = tx0; tx <= tx1; ++tx)
        for (int ty = ty0; ty <= ty1; ++ty) flags[tx * tiles_y + ty] = 1;
}

}  // namespace

void launch_tile_flags(const int *list0, const int *cnt0, const int *list1, const int *cnt1, int ncells, int nx,
                       int ny, int *flags, hipStream_t s) {
    const int tx = (nx + kSplitTile - 1) / kSplitTile, ty = (ny + kSplitTile - 1) / kSplitTile;
    hipLaunchKernelGGL(tile_flag_clear_kernel, dim3((tx * ty + 255) / 256), dim3(256), 0, s, flags, tx * ty);
    hipLaunchKernelGGL(tile_flag_mark_kernel, dim3((ncells + 255) / 256), dim3(256), 0, s, list0, cnt0, list1, cnt1,
                       ncells, ny + 4, tx, ty, flags);
}

void launch_ghost_fill(const GridArgs &g, hipStream_t s) {
    if (g.init_cond != 2) return;
    const int nxs = 2 * g.ny * g.nm, nys = g.nx * 2 * g.nm;
    hipLaunchKernelGGL(ghost_x_kernel, dim3((nxs + kBlock - 1) / kBlock), dim3(kBlock), 0, s, g);
    hipLaunchKernelGGL(ghost_y_kernel, dim3((nys + kBlock - 1) / kBlock), dim3(kBlock), 0, s, g);
}

#define MNC_NM_SWITCH(NMV, CALL) \
    switch (NMV) {               \
    case 1: CALL(1); break;      \
    case 3: CALL(3); break;      \
    case 6: CALL(6); break;      \
    case 10: CALL(10); break;    \
    case 15: CALL(15); break;    \
    case 21: CALL(21); break;    \
    case 28: CALL(28); break;    \
    case 36: CALL(36); break;    \
    case 45: CALL(45); break;    \
    default: return false;       \
    }

void launch_ansatz(const GridArgs &g, int q0, int nqc, hipStream_t s) {
    auto f = [&]() -> bool {
#define CALLA(N) launch_ansatz_t<N>(g, q0, nqc, s)
        MNC_NM_SWITCH(g.nm, CALLA)
#undef CALLA
        return true;
    };
    f();
}

bool launch_flux_fused(const GridArgs &g, int tile, int stage, double dt, hipStream_t s) {
#define CALLX(N) launch_fused_t<N>(g, tile, stage, dt, s)
    MNC_NM_SWITCH(g.nm, CALLX)
#undef CALLX
    return true;
}

bool launch_flux_euler(const GridArgs &g, int q0, int nqc, int stage, double dt, bool first_chunk, bool last_chunk,
                       hipStream_t s) {
#define CALLF(N) launch_flux_t<N>(g, q0, nqc, stage, dt, first_chunk, last_chunk, s)
    MNC_NM_SWITCH(g.nm, CALLF)
#undef CALLF
    return true;
}

}  // namespace mnc
