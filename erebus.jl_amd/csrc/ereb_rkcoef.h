// ereb_rkcoef.h -- the RK4 stage-velocity coefficient tables, filled by a
// kernel of their own (ereb_markers.hip) or beside the sort's placement
// (ereb_sort.hip).
#pragma once
#include "ereb_internal.h"

namespace ereb {

// RK4 stage velocities as quadratics, prepared once per step
// (k_rk4_coef, or beside the sort's placement in the transfer step).
// On the Vx grid (E:5057-5091) the stage velocity in cell (i, j) is
//   v = v_i(fx) + fy (v_{i+1}(fx) - v_i(fx)),
//   v_r(fx) = a_r + fx (b_r - a_r) + 0.5 (fx - 0.5)^2 d_r,
// a_r = v[r, j], b_r = v[r, j+1], and d_r the second difference
// v[r, c-1] - 2 v[r, c] + v[r, c+1] (the reference's association) at the
// correction's centre column c = j for fx < 0.5 ("left" half), c = j + 1
// otherwise, zero where the reference skips the correction (c == 1 left,
// c == Nx right, i.e. outside 2 <= c <= Nx-1).  In the fluid loop the
// centre of the first row's left-half correction is read from vx (E:5173).
// Expanding 0.5 (fx - 0.5)^2 = 0.125 - 0.5 fx + 0.5 fx^2, each half of each
// cell is v = P(fx) + fy Q(fx) with
//   P = (a_i + d_i/8) + fx ((b_i - a_i) - d_i/2) + fx^2 (d_i/2),
//   Q = the same of row i+1 minus P,
// six coefficients [P0 P1 P2 Q0 Q1 Q2]; the Vy grid (E:5093-5127) is the
// transpose (quadratic in fy, linear in fx).  Table layout: per cell of the
// (Ny1, Nx1) node numbering, 12 doubles (left half, then right half), so a
// stage reads its half with three 16-byte loads; four tables (Vx and Vy of
// the solid and of the fluid loop).
constexpr int RKC = 12;  // doubles per cell and table

struct RKCoefArgs {
    int Nx, Ny;
    const double *vx, *vy, *vxf, *vyf;
    double *cxs, *cys, *cxf, *cyf;  // tables: Vx solid, Vy solid, Vx fluid, Vy fluid
};

// second difference of g along a line at index k with stride s, if the
// centre's position c lies in [2, n-1] (else the correction is skipped)
__device__ __forceinline__ double d2(const double* __restrict__ q, const double* __restrict__ ctr,
                                     int k, int s, int c, int n) {
    return (c >= 2 && c <= n - 1) ? (q[k - s] - 2.0 * ctr[k]) + q[k + s] : 0.0;
}

// coefficients of one half: rows (a0, b0, d0) and (a1, b1, d1) along the
// quadratic direction
__device__ __forceinline__ void rk_half(double* __restrict__ out, double a0, double b0,
                                        double d0, double a1, double b1, double d1) {
    const double p0 = a0 + 0.125 * d0, p1 = (b0 - a0) - 0.5 * d0, p2 = 0.5 * d0;
    const double r0 = a1 + 0.125 * d1, r1 = (b1 - a1) - 0.5 * d1, r2 = 0.5 * d1;
    out[0] = p0;
    out[1] = p1;
    out[2] = p2;
    out[3] = r0 - p0;
    out[4] = r1 - p1;
    out[5] = r2 - p2;
}

// One thread per cell of one table, cells in table order
// (k = (j - 1) Ny1 + (i - 1)): the thread loads the cell's velocity
// neighbourhood once and evaluates both halves; the workgroup's 256 cells
// (24 KB of coefficients) are assembled in LDS and written with consecutive
// 16-byte stores.
constexpr int RKCOEF_CELLS = 256;

// bx: block of RKCOEF_CELLS cells, t: table; sh: RKCOEF_CELLS * RKC doubles of LDS
// (A by value: of a reference's four tables the compiler picks one through
// scratch memory, 40 bytes a lane, a third more writes than the tables'; the
// launch with the placement at 141 x 141 nodes took 8.6 us, 5.9 now)
__device__ __forceinline__ void rk4_coef_block(RKCoefArgs A, int bx, int t,
                                               double* __restrict__ sh) {
    const int R = A.Ny + 1;
    const int N = R * (A.Nx + 1);
    const int b0 = bx * RKCOEF_CELLS;
    const int k = b0 + (int)threadIdx.x;
    // t: 0 Vx solid, 1 Vy solid, 2 Vx fluid, 3 Vy fluid
    const bool xg = (t & 1) == 0, fluid = t >= 2;
    double c[RKC];
#pragma unroll
    for (int q = 0; q < RKC; ++q) c[q] = 0.0;
    if (k < N) {
        const int i = k % R + 1, j = k / R + 1;
        const int k1 = k + 1, kR = k + R, kR1 = k + R + 1;
        if (xg && i <= A.Ny && j <= A.Nx - 1) {
            // Vx cell (i, j): rows i, i+1 of columns j, j+1; centre column j
            // (left half) or j+1 (right half); the fluid loop's first-row
            // left-half centre is read from vx (E:5173)
            const double* v = fluid ? A.vxf : A.vx;
            const double a0 = v[k], b0v = v[kR], a1 = v[k1], b1 = v[kR1];
            rk_half(c, a0, b0v, d2(v, fluid ? A.vx : v, k, R, j, A.Nx), a1, b1,
                    d2(v, v, k1, R, j, A.Nx));
            rk_half(c + 6, a0, b0v, d2(v, v, kR, R, j + 1, A.Nx), a1, b1,
                    d2(v, v, kR1, R, j + 1, A.Nx));
        } else if (!xg && i <= A.Ny - 1 && j <= A.Nx) {
            // Vy cell (i, j): rows i, i+1 of columns j, j+1; centre row i
            // (upper half) or i+1 (lower half)
            const double* v = fluid ? A.vyf : A.vy;
            const double a0 = v[k], b0v = v[k1], a1 = v[kR], b1 = v[kR1];
            rk_half(c, a0, b0v, d2(v, v, k, 1, i, A.Ny), a1, b1, d2(v, v, kR, 1, i, A.Ny));
            rk_half(c + 6, a0, b0v, d2(v, v, k1, 1, i + 1, A.Ny), a1, b1,
                    d2(v, v, kR1, 1, i + 1, A.Ny));
        }
    }
#pragma unroll
    for (int q = 0; q < RKC; q += 2)
        *(double2*)(sh + threadIdx.x * RKC + q) = make_double2(c[q], c[q + 1]);
    __syncthreads();
    double* out = t == 0 ? A.cxs : (t == 1 ? A.cys : (t == 2 ? A.cxf : A.cyf));
    const int npiece = min(RKCOEF_CELLS, N - b0) * (RKC / 2);
    for (int p = threadIdx.x; p < npiece; p += RKCOEF_CELLS)
        *(double2*)(out + (size_t)b0 * RKC + 2 * p) = *(const double2*)(sh + 2 * p);
}

// the tables' arguments and blocks per table (ereb_markers.hip)
RKCoefArgs rk4_coef_args(ereb_ctx* c);
inline unsigned rk4_coef_blocks(const ereb_ctx* c) {
    return (unsigned)(((int64_t)c->Ny1 * c->Nx1 + RKCOEF_CELLS - 1) / RKCOEF_CELLS);
}

}  // namespace ereb
