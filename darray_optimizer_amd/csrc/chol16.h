// Cholesky of one 16 x 16 FP64 block by one wave, shared by the CholeskyQR
// Cholesky (small_spd.h) and the diagonal blocks of the blocked one (dense.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "mfma_tile.h"

namespace {

__device__ __forceinline__ double readlane_d(double v, int lane) {
    int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
    int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
    return __hiloint2double(hi, lo);
}

// Orders LDS traffic of one wave (no workgroup barrier: waves are independent).
// Waits for LDS traffic only (s_waitcnt lgkmcnt(0) with vmcnt / expcnt left at
// their maxima), so prefetched global loads stay in flight across it.
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_wave_barrier();
}

// The values of the four 16-lane rows at the lane's column: out[g] = v of lane
// 16 g + (lane & 15).
__device__ __forceinline__ void gather_rows(double v, double (&out)[4]) {
    const unsigned lo = (unsigned)__double2loint(v), hi = (unsigned)__double2hiint(v);
    const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);  // rows 0022, 1133
    const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    const auto l02 = __builtin_amdgcn_permlane32_swap(l[0], l[0], false, false);
    const auto h02 = __builtin_amdgcn_permlane32_swap(h[0], h[0], false, false);
    const auto l13 = __builtin_amdgcn_permlane32_swap(l[1], l[1], false, false);
    const auto h13 = __builtin_amdgcn_permlane32_swap(h[1], h[1], false, false);
    out[0] = __hiloint2double((int)h02[0], (int)l02[0]);
    out[1] = __hiloint2double((int)h13[0], (int)l13[0]);
    out[2] = __hiloint2double((int)h02[1], (int)l02[1]);
    out[3] = __hiloint2double((int)h13[1], (int)l13[1]);
}

// 1/sqrt(piv): hardware estimate and two Newton steps; INF: 0 for infinity (NaN
// without it).
template <bool INF>
__device__ __forceinline__ double rsqrt_newton(double piv) {
    const double hp = 0.5 * (INF ? fmin(piv, 0x1.fffffffffffffp+1023) : piv);
    double y = __builtin_amdgcn_rsq(piv);
    y = fma(y, fma(-hp * y, y, 0.5), y);
    return fma(y, fma(-hp * y, y, 0.5), y);
}

// Cholesky of a 16 x 16 block in MFMA accumulator layout (d[r] of lane (g, li):
// row g + 4r, column li) by one wave, in four steps of four rows; on return d
// holds U (entries below the diagonal are whatever the updates leave there).
// Rows 4b .. 4b+3 are d[b] of the four lane groups.  Every lane factors the
// 4 x 4 diagonal block for itself (uniform values) and solves the four rows at
// its own column, so the chain of square roots crosses no lanes; then d[b] =
// the lane's row is the operand of one MFMA that updates all later rows (rows
// up to 4b+3 masked).  An FP64 MFMA is a chain of FMAs in ascending k, so each
// element gets fma(-u_k, u_k', a) once per step k, as column by column.
// Returns 0, or the 1-based step of the first pivot p with !(p > tol) among
// the first nreal.  INF: an infinite pivot gives a row of zeros with inf / inf on
// the diagonal, which stays there (finished columns are masked too); without it
// the row and the pivots after it are NaN.  About 450 cycles per four rows; a
// step per row with broadcasts of the row took 300 per row.
template <bool INF = false>
__device__ __forceinline__ int chol16(dh_d4& d, int g, int li, int nreal, double tol) {
    int bad = 0;  // no early exit: what follows a failed pivot is not used
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        double a[4];
        gather_rows(d[b], a);
        double m[4][4];  // the diagonal block, upper part, uniform
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int c = r; c < 4; ++c) m[r][c] = readlane_d(d[b], 16 * r + 4 * b + c);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int kk = 4 * b + r;
            bad = bad == 0 && kk < nreal && !(m[r][r] > tol) ? kk + 1 : bad;
            const double y = rsqrt_newton<INF>(m[r][r]);
            a[r] *= y;
#pragma unroll
            for (int c = r + 1; c < 4; ++c) m[r][c] *= y;
#pragma unroll
            for (int i = r + 1; i < 4; ++i) {
#pragma unroll
                for (int c = i; c < 4; ++c) m[i][c] = fma(-m[r][i], m[r][c], m[i][c]);
                a[i] = fma(-m[r][i], a[r], a[i]);
            }
        }
        double u = a[0];
        u = g == 1 ? a[1] : u;
        u = g == 2 ? a[2] : u;
        u = g == 3 ? a[3] : u;
        d[b] = u;
        const bool later = li > 4 * b + 3;
        if (b < 3) d = Mfma<double>::op(later ? -u : 0.0, INF && !later ? 0.0 : u, d);
    }
    return bad;
}

}  // namespace
