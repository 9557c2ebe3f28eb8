// Nystrom factor of the range finder (the consumer step of testsvm.cpp:126-177)
// and the one-sided Jacobi SVD it runs on.
//
// Reference: C = Q^T (K Q) by tc_gemm (testsvm.cpp:126-137), its singular
// values by sgesvd_ on the host (DArray::svd, lapack_like.h:388-413), then
// Z = Q diag(S) (testsvm.cpp:146-172) -- which drops the singular vectors.
// Here C = (Q^T W + W^T Q)/2 with W = K Q from dh_lra, its eigenpairs from a
// one-sided (Hestenes) Jacobi SVD on the device in FP64, and
// Z = Q V_k diag(sqrt(max(lam_k, 0))), so Z Z^T = Q V_k Lam_k V_k^T Q^T is
// the rank-k truncation of Q Q^T K Q Q^T.
//
// Jacobi: all column pairs of one round of a round-robin tournament are
// disjoint, and from one round to the next a column only moves to a
// neighbouring pair.  So a workgroup that holds a run of neighbouring pairs in
// LDS runs several rounds by itself (jacobi_rounds_kernel), and V follows
// once per sweep from a log of the rotations (jacobi_apply_kernel).  Columns
// too long for that take one launch per round (jacobi_round_kernel).
// A device flag records whether a sweep rotated anything; the rounds of later
// sweeps return at once after a sweep that did not, and the host reads the
// flag once per sweep.
#include <algorithm>
#include <cmath>

#include "dh_common.h"

namespace {

constexpr double kJacobiTol = 1e-14;  // rotate when |a_p.a_q| > tol |a_p| |a_q|
constexpr int kMaxSweeps = 60;

// Player at position pos of a round, round <= N - 1 (so one subtraction is the modulus).
__device__ __forceinline__ int rr_player(int pos, int round, int N) {
    const int x = pos - 1 + round;
    return pos == 0 ? 0 : 1 + (x >= N - 1 ? x - (N - 1) : x);
}

// Sum over the wave's 64 lanes, the same value in every lane: the butterfly
// over lane distances 32, 16, 8, 4, 2, 1 with register permutes only.  After
// distance 8 a lane's value depends on its index modulo 8 alone (then 4, 2),
// so a rotation within the 16-lane row stands for the exchange.
__device__ __forceinline__ double join_halves(unsigned lo, unsigned hi) {
    return __hiloint2double((int)hi, (int)lo);
}
template <int CTRL>
__device__ __forceinline__ double add_dpp(double v) {
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, false);
    return v + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double read_lane(double v, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}
__device__ __forceinline__ double add_swap32(double a, double b) {
    const auto l = __builtin_amdgcn_permlane32_swap((unsigned)__double2loint(a),
                                                    (unsigned)__double2loint(b), false, false);
    const auto h = __builtin_amdgcn_permlane32_swap((unsigned)__double2hiint(a),
                                                    (unsigned)__double2hiint(b), false, false);
    return join_halves(l[0], h[0]) + join_halves(l[1], h[1]);
}
__device__ __forceinline__ double add_swap16(double a, double b) {
    const auto l = __builtin_amdgcn_permlane16_swap((unsigned)__double2loint(a),
                                                    (unsigned)__double2loint(b), false, false);
    const auto h = __builtin_amdgcn_permlane16_swap((unsigned)__double2hiint(a),
                                                    (unsigned)__double2hiint(b), false, false);
    return join_halves(l[0], h[0]) + join_halves(l[1], h[1]);
}
__device__ __forceinline__ double wave_sum(double v) {
    v = add_swap32(v, v);
    v = add_swap16(v, v);
    v = add_dpp<0x128>(v);  // row_ror:8
    v = add_dpp<0x124>(v);  // row_ror:4
    v = add_dpp<0x122>(v);  // row_ror:2
    return add_dpp<0x121>(v);  // row_ror:1
}

// The sums of a, b and c over the wave's lanes, in the order of wave_sum but
// with the three sharing its steps: after the exchange over lane distance 32 the
// lower half works on a and the upper half on b, after distance 16 the odd
// rows work on c (7 additions and 14 permutes instead of 18 and 36).
__device__ __forceinline__ void wave_sum3(double& a, double& b, double& c) {
    double v = add_swap16(add_swap32(a, b), add_swap32(c, c));  // rows: a, c, b, c
    v = add_dpp<0x128>(v);
    v = add_dpp<0x124>(v);
    v = add_dpp<0x122>(v);
    v = add_dpp<0x121>(v);
    a = read_lane(v, 0);
    b = read_lane(v, 32);
    c = read_lane(v, 16);
}

// Square root and reciprocal, correctly rounded as the IEEE forms, of values
// in [1, 2^1000): hardware estimate, Newton steps, a residual correction; no
// scaling and no special cases (half of the IEEE forms' instructions).
__device__ __forceinline__ double sqrt_ge1(double w) {
    const double y = __builtin_amdgcn_rsq(w);
    double g = w * y, hf = 0.5 * y;
    const double r = fma(-hf, g, 0.5);
    g = fma(g, r, g);
    hf = fma(hf, r, hf);
    g = fma(fma(-g, g, w), hf, g);
    return fma(fma(-g, g, w), hf, g);
}
__device__ __forceinline__ double recip_ge1(double w) {
    double r = __builtin_amdgcn_rcp(w);
    r = fma(r, fma(-w, r, 1.0), r);
    r = fma(r, fma(-w, r, 1.0), r);
    return fma(fma(-w, r, 1.0), r, r);
}

// Rutishauser's rotation (c, s) of a pair with squared norms al, be and dot
// product ga: the smaller root t of t^2 + 2 zeta t - 1 = 0.  False when the
// pair counts as orthogonal ((c, s) is then of no use: the angle is computed
// beside the test, not after it).  Every rounding matters here: a pair of
// equal norms turns by +45 or -45 degrees on the last bit of zeta, which
// decides the sign of a singular vector, so the operations are fixed (FMAs
// written out) and the roots correctly rounded.  |zeta| is held below 2^490,
// past which t is 0 to working precision.
__device__ __forceinline__ bool jacobi_angle(double al, double be, double ga, double tol, double& c,
                                             double& s) {
    const double zeta = (be - al) / (2.0 * ga);
    const double az = fmin(fabs(zeta), 0x1p490);
    double t = recip_ge1(az + sqrt_ge1(fma(az, az, 1.0)));
    t = zeta >= 0.0 ? t : -t;
    c = recip_ge1(sqrt_ge1(fma(t, t, 1.0)));
    s = c * t;
    return fabs(ga) > tol * sqrt(al * be);
}

__device__ __forceinline__ void rotate(double c, double s, double x, double y, double& p,
                                       double& q) {
    p = fma(c, x, -(s * y));
    q = fma(s, x, c * y);
}

// One round, a wave per pair.  flags[0]: a pair rotated in the current sweep;
// flags[1]: converged.
__global__ __launch_bounds__(64) void jacobi_round_kernel(int m, int n, int N, int round,
                                                          double* __restrict__ A, int lda,
                                                          double* __restrict__ V, int ldv,
                                                          double tol, int* __restrict__ flags) {
    if (flags[1]) return;
    int p = rr_player(blockIdx.x, round, N), q = rr_player(N - 1 - blockIdx.x, round, N);
    if (p >= n || q >= n) return;  // the padding player of an odd n
    if (p > q) {
        const int t = p;
        p = q;
        q = t;
    }
    double* ap = A + (size_t)p * lda;
    double* aq = A + (size_t)q * lda;
    const int lane = threadIdx.x;
    double al = 0.0, be = 0.0, ga = 0.0;
    for (int e = lane; e < m; e += 64) {
        const double x = ap[e], y = aq[e];
        al = fma(x, x, al);
        be = fma(y, y, be);
        ga = fma(x, y, ga);
    }
    wave_sum3(al, be, ga);
    double c, s;
    if (!jacobi_angle(al, be, ga, tol, c, s)) return;
    for (int e = lane; e < m; e += 64) {
        const double x = ap[e], y = aq[e];
        rotate(c, s, x, y, ap[e], aq[e]);
    }
    double* vp = V + (size_t)p * ldv;
    double* vq = V + (size_t)q * ldv;
    for (int e = lane; e < n; e += 64) {
        const double x = vp[e], y = vq[e];
        rotate(c, s, x, y, vp[e], vq[e]);
    }
    if (lane == 0) atomicOr(&flags[0], 1);
}

// Rounds [r0, r0 + T) on the columns of `own` neighbouring pairs (cells) per
// workgroup.  Cell b of a round holds the players at positions b and N-1-b;
// from round to round the upper players move one cell down, the lower ones
// one cell up, turning round at both ends, so the columns of a cell T rounds
// later come from the cells at most T away.  The workgroup therefore loads
// its own cells and T more on each side, and round t covers the loaded cells
// but for t at each open side; the outer ones are computed by the neighbour
// too, with the same operations on the same values.  Columns stay in the LDS
// slot of their first position (the cell of a later round finds them by
// index); own cells are written to Aout, another buffer than Ain unless one
// workgroup holds every cell.  The rotations of own cells go to
// cs[round * N/2 + cell] for V.
//
// What bounds it: the chain of one round (LDS reads, three wave sums, two
// square roots and three divisions, LDS writes, a barrier), about two cells
// per wave at 32 cells; a launch per round spent most of its time on the
// launch and on re-reading its columns.  Arithmetic and order are those of
// jacobi_round_kernel.
constexpr int kJacWaves = 16;
constexpr int kJacDoubles = 19968;  // columns held by a workgroup: 156 KB of LDS

template <int E>  // ceil(m / 64); columns are padded with zeros to 64 E in LDS
__global__ __launch_bounds__(kJacWaves * 64) void jacobi_rounds_kernel(
    int m, int n, int N, int r0, int T, int own, const double* Ain, int ldi, double* Aout, int ldo,
    double2* __restrict__ cs, double tol, int* __restrict__ flags) {
    __shared__ double col[kJacDoubles];
    if (flags[1]) return;
    constexpr int P = 64 * E;  // LDS pitch of a column
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int half = N / 2;
    const int own0 = blockIdx.x * own, own1 = min(half, own0 + own);
    const int lo = max(0, own0 - T), hi = min(half, own1 + T);
    // Slot of the column at position pos of round r0 + t: positions move as
    // players do, so it began at position rr_player(pos, t).
    auto slot = [&](int pos, int t) {
        const int p0 = rr_player(pos, t, N);
        const int q0 = N - 1 - p0;
        return 2 * (min(p0, q0) - lo) + (p0 < q0 ? 0 : 1);
    };
    // Four columns per wave and step, all loads before the first LDS store
    // (clamped addresses: a load under a branch is waited for by itself).  The
    // padding player of an odd n is a zero column: it never rotates.
    for (int cb = 2 * lo + wave; cb < 2 * hi; cb += 4 * kJacWaves) {
        double v[4][E];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int c = min(cb + k * kJacWaves, 2 * hi - 1);
            const int pl = rr_player((c & 1) ? N - 1 - (c >> 1) : (c >> 1), r0, N);
            const double* src = Ain + (size_t)min(pl, n - 1) * ldi;
#pragma unroll
            for (int u = 0; u < E; ++u) {
                v[k][u] = src[min(lane + 64 * u, m - 1)];
                if (pl >= n || (u + 1 == E && lane + 64 * u >= m)) v[k][u] = 0.0;
            }
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int c = cb + k * kJacWaves;
            if (c < 2 * hi)
#pragma unroll
                for (int u = 0; u < E; ++u) col[(c - 2 * lo) * P + lane + 64 * u] = v[k][u];
        }
    }
    __syncthreads();
    int rotated = 0;
    for (int t = 0; t < T; ++t) {
        const int c0 = lo == 0 ? 0 : lo + t, c1 = hi == half ? half : hi - t;
        for (int b = c0 + wave; b < c1; b += kJacWaves) {
            const int s0 = slot(b, t), s1 = slot(N - 1 - b, t);
            const bool swap = rr_player(b, r0 + t, N) > rr_player(N - 1 - b, r0 + t, N);
            double* ap = col + (swap ? s1 : s0) * P + lane;
            double* aq = col + (swap ? s0 : s1) * P + lane;
            double x[E], y[E], al = 0.0, be = 0.0, ga = 0.0;
#pragma unroll
            for (int u = 0; u < E; ++u) {
                x[u] = ap[64 * u];
                y[u] = aq[64 * u];
            }
#pragma unroll
            for (int u = 0; u < E; ++u) {
                al = fma(x[u], x[u], al);
                be = fma(y[u], y[u], be);
                ga = fma(x[u], y[u], ga);
            }
            wave_sum3(al, be, ga);
            double c, s;
            const bool rot = __builtin_amdgcn_readfirstlane(jacobi_angle(al, be, ga, tol, c, s));
            if (rot) {
#pragma unroll
                for (int u = 0; u < E; ++u) rotate(c, s, x[u], y[u], ap[64 * u], aq[64 * u]);
                rotated = 1;
            }
            if (lane == 0 && b >= own0 && b < own1)
                cs[(size_t)(r0 + t) * half + b] = make_double2(c, rot ? s : 0.0);
        }
        __syncthreads();
    }
    // Own cells of round r0 + T: the player and the slot of each position.
    for (int c = 2 * own0 + wave; c < 2 * own1; c += kJacWaves) {
        const int pos = (c & 1) ? N - 1 - (c >> 1) : (c >> 1);
        const int pl = rr_player(pos, r0 + T, N);
        if (pl >= n) continue;
        const double* src = col + slot(pos, T) * P + lane;
        double* dst = Aout + (size_t)pl * ldo + lane;
#pragma unroll
        for (int u = 0; u < E; ++u)
            if (u + 1 < E || lane + 64 * u < m) dst[64 * u] = src[64 * u];
    }
    if (rotated && lane == 0) atomicOr(&flags[0], 1);
}

// V := V * (the rotations of one sweep, from cs): rows are independent, so a
// workgroup keeps kJacRows rows of V (every column) in LDS and runs all
// N - 1 rounds, a thread per (cell, row); the next round's (c, s) are loaded
// a round ahead.
constexpr int kJacRows = 4;
constexpr int kJacApplyMaxN = 1024;

__global__ __launch_bounds__(1024) void jacobi_apply_kernel(int n, int N,
                                                            const double2* __restrict__ cs,
                                                            double* __restrict__ V, int ldv,
                                                            const int* __restrict__ rotated) {
    __shared__ double v[kJacApplyMaxN * kJacRows];  // v[column][row]
    if (*rotated == 0) return;
    const int half = N / 2, row0 = blockIdx.x * kJacRows;
    for (int e = threadIdx.x; e < n * kJacRows; e += blockDim.x) {
        const int r = e % kJacRows, j = e / kJacRows;
        v[e] = row0 + r < n ? V[row0 + r + (size_t)j * ldv] : 0.0;
    }
    const int r = threadIdx.x % kJacRows, b0 = threadIdx.x / kJacRows;
    const int step = blockDim.x / kJacRows;
    // Rotations of the thread's first cell, kAhead rounds ahead (a global load
    // takes longer than a round).
    constexpr int kAhead = 8;
    const int bl = min(b0, half - 1);
    auto fetch = [&](int round) { return cs[(size_t)min(round, N - 2) * half + bl]; };
    double2 nx[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k) nx[k] = fetch(k);
    __syncthreads();
    auto apply = [&](int round, int b, double2 w) {
        if (w.y == 0.0) return;  // not rotated (or a rotation by nothing)
        int p = rr_player(b, round, N), q = rr_player(N - 1 - b, round, N);
        if (p > q) {
            const int t = p;
            p = q;
            q = t;
        }
        const double x = v[p * kJacRows + r], y = v[q * kJacRows + r];
        rotate(w.x, w.y, x, y, v[p * kJacRows + r], v[q * kJacRows + r]);
    };
    for (int r0 = 0; r0 < N - 1; r0 += kAhead) {
#pragma unroll
        for (int k = 0; k < kAhead; ++k) {
            const int round = r0 + k;
            if (round < N - 1) {  // uniform
                if (b0 < half) apply(round, b0, nx[k]);
                nx[k] = fetch(round + kAhead);
                for (int b = b0 + step; b < half; b += step)
                    apply(round, b, cs[(size_t)round * half + b]);
                __syncthreads();
            }
        }
    }
    for (int e = threadIdx.x; e < n * kJacRows; e += blockDim.x) {
        const int rr = e % kJacRows, j = e / kJacRows;
        if (row0 + rr < n) V[row0 + rr + (size_t)j * ldv] = v[e];
    }
}

// words[0]: a pair rotated in the current sweep; [1]: converged; [2]: sweeps
// run; [4 + s % 4]: sweep s rotated a pair (for the update of V).
// End of sweep s: converged if nothing rotated; clear the rotation flag.
__global__ void jacobi_sweep_end_kernel(int* __restrict__ words, int s) {
    if (threadIdx.x != 0) return;
    const int rotated = words[1] ? 0 : words[0];
    words[4 + s % 4] = rotated;
    if (words[1]) return;
    words[2] += 1;
    if (!rotated) words[1] = 1;
    words[0] = 0;
}

__global__ void jacobi_init_words_kernel(int* __restrict__ words) {
    if (threadIdx.x < 8) words[threadIdx.x] = 0;
}

// V = I (n x n).
__global__ __launch_bounds__(256) void identity_kernel(int n, double* __restrict__ V, int ldv) {
    const size_t total = (size_t)n * n;
    for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < total;
         e += (size_t)gridDim.x * 256) {
        const int i = (int)(e % n), j = (int)(e / n);
        V[i + (size_t)j * ldv] = (i == j) ? 1.0 : 0.0;
    }
}

// key[j] = |A[:, j]| (mode 0) or V[:, j] . A[:, j] (mode 1: the signed
// eigenvalue when A = C V for symmetric C); one wave per column.
__global__ __launch_bounds__(256) void column_key_kernel(int m, int n, const double* __restrict__ A,
                                                         int lda, const double* __restrict__ V,
                                                         int ldv, int mode,
                                                         double* __restrict__ key) {
    const int j = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (j >= n) return;
    const double* a = A + (size_t)j * lda;
    double s = 0.0;
    if (mode == 0) {
        for (int e = lane; e < m; e += 64) s += a[e] * a[e];
    } else {
        const double* v = V + (size_t)j * ldv;
        for (int e = lane; e < m; e += 64) s += v[e] * a[e];
    }
    s = wave_sum(s);
    if (lane == 0) key[j] = mode == 0 ? sqrt(s) : s;
}

// ord[rank] = j for keys in descending order, ties by column index (one
// workgroup; rank by counting, n <= a few thousand).
__global__ __launch_bounds__(1024) void rank_desc_kernel(int n, const double* __restrict__ key,
                                                         int* __restrict__ ord) {
    for (int j = threadIdx.x; j < n; j += 1024) {
        const double kj = key[j];
        int r = 0;
        for (int i = 0; i < n; ++i) {
            const double ki = key[i];
            r += (ki > kj) || (ki == kj && i < j);
        }
        ord[r] = j;
    }
}

// dst[:, j] = scale_j * src[:, ord[j]] for j < cols (m rows); scale_j =
// sqrt(max(key[ord[j]], 0)) when sqrt_scale, else 1; keys_out[j] = key[ord[j]].
__global__ __launch_bounds__(256) void gather_columns_kernel(
    int m, int cols, const double* __restrict__ src, int lds, const int* __restrict__ ord,
    const double* __restrict__ key, int sqrt_scale, double* __restrict__ dst, int ldd,
    double* __restrict__ keys_out) {
    const size_t total = (size_t)m * cols;
    for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < total;
         e += (size_t)gridDim.x * 256) {
        const int i = (int)(e % m), j = (int)(e / m);
        const int o = ord[j];
        double sc = 1.0;
        if (sqrt_scale) {
            const double v = key[o];
            sc = v > 0.0 ? sqrt(v) : 0.0;
        }
        dst[i + (size_t)j * ldd] = sc * src[i + (size_t)o * lds];
        if (i == 0 && keys_out) keys_out[j] = key[o];
    }
}

// C = (C + C^T) / 2 on the n x n C (ld ldc).
__global__ __launch_bounds__(256) void symmetrize_kernel(int n, double* __restrict__ C, int ldc) {
    const size_t total = (size_t)n * n;
    for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < total;
         e += (size_t)gridDim.x * 256) {
        const int i = (int)(e % n), j = (int)(e / n);
        if (i >= j) continue;
        const double s = 0.5 * (C[i + (size_t)j * ldc] + C[j + (size_t)i * ldc]);
        C[i + (size_t)j * ldc] = s;
        C[j + (size_t)i * ldc] = s;
    }
}

__global__ __launch_bounds__(256) void copy_cols_kernel(int m, int n, const double* __restrict__ src,
                                                        int lds, double* __restrict__ dst, int ldd) {
    const size_t total = (size_t)m * n;
    for (size_t e = (size_t)blockIdx.x * 256 + threadIdx.x; e < total;
         e += (size_t)gridDim.x * 256) {
        const int i = (int)(e % m), j = (int)(e / m);
        dst[i + (size_t)j * ldd] = src[i + (size_t)j * lds];
    }
}

int grid_for(size_t total) { return (int)std::min<size_t>((total + 255) / 256, 4096); }

// How the rounds of a sweep are grouped: `own` cells per workgroup, at most T
// rounds per launch, `launches` per sweep.  own = 0: one launch per round, for
// columns or orders that LDS does not hold and for a single pair.  A round
// costs about 0.8 us + 0.25 us per four cells of a workgroup, a launch with its
// loads and stores 5 us.  So up to 20 cells are one workgroup and one launch per
// sweep (order 16 0.47 -> 0.23 ms, 4 0.14 ms either way, 2 0.09 ms and 0.14 in one
// workgroup), and larger orders are cut into many small workgroups that share
// cells: 4 own cells and 12 rounds, 28 cells at the first (order 272, n = 65536: 26.6
// -> 11.2 ms per factor).  Long columns lower T until the cells fit in LDS.
// `launches` is even there, so that a sweep ends in the buffer that it began in.
struct JacobiPlan {
    int own = 0, T = 0, launches = 0;
};

JacobiPlan jacobi_plan(int m, int n) {
    JacobiPlan p;
    const int N = n + (n & 1), half = N / 2;
    if (m > 512 || N > kJacApplyMaxN || N == 2) return p;
    const int cap = kJacDoubles / (128 * dh_cdiv(m, 64));  // cells that fit in LDS (>= 19)
    if (half <= std::min(cap, 20)) {
        p.own = half;
        p.T = N - 1;
        p.launches = 1;
        return p;
    }
    p.own = 4;
    p.T = (std::min(cap, 28) - p.own) / 2;
    p.launches = dh_cdiv(N - 1, p.T);
    p.launches += p.launches & 1;
    return p;
}

// Doubles of work space that jacobi_sweeps wants beside A and V: a second
// buffer for A's columns and the rotations of two sweeps, or nothing where a
// round is a launch.
size_t jacobi_work_doubles(int m, int n) {
    if (jacobi_plan(m, n).own == 0) return 0;
    const size_t N = n + (n & 1);
    return (size_t)m * n + 2 * (N - 1) * N + 2;
}

int launch_rounds(dh_handle_t h, int m, int n, int N, int r0, int T, int own, const double* Ain,
                  int ldi, double* Aout, int ldo, double2* cs, int* words) {
    const int grid = dh_cdiv(N / 2, own);
#define DH_JAC(E)                                                                              \
    case E:                                                                                    \
        jacobi_rounds_kernel<E><<<grid, kJacWaves * 64, 0, h->stream>>>(                       \
            m, n, N, r0, T, own, Ain, ldi, Aout, ldo, cs, kJacobiTol, words);                  \
        break;
    switch (dh_cdiv(m, 64)) {
        DH_JAC(1)
        DH_JAC(2)
        DH_JAC(3)
        DH_JAC(4)
        DH_JAC(5)
        DH_JAC(6)
        DH_JAC(7)
        default:
        DH_JAC(8)
    }
#undef DH_JAC
    DH_CHECK_LAUNCH();
    return 0;
}

// Jacobi sweeps on A (m x n) accumulating V (n x n, set to I here); flags and
// the sweep counter live in `words` (8 ints of device memory), `work` holds
// jacobi_work_doubles(m, n).  *sweeps_out receives the sweeps run, or -1 if
// kMaxSweeps did not converge.  Where a sweep is several launches V's update
// runs on the handle's second stream beside the next sweep (1 ms of 11 at order
// 272), and the handle's stream waits for it before the call goes on; where it
// is one launch the events would cost more (orders up to 16: 0.25 ms against 0.14).
int jacobi_sweeps(dh_handle_t h, int m, int n, double* A, int lda, double* V, int ldv,
                  double* work, int* words, int* sweeps_out) {
    hipStream_t s = h->stream;
    identity_kernel<<<grid_for((size_t)n * n), 256, 0, s>>>(n, V, ldv);
    DH_CHECK_LAUNCH();
    jacobi_init_words_kernel<<<1, 64, 0, s>>>(words);
    DH_CHECK_LAUNCH();
    *sweeps_out = 0;
    if (n < 2) return 0;
    int* host = dh_host_status(h);
    if (!host) return dh_fail(DH_ERR_ALLOC, "dh_gesvj: pinned status words unavailable");
    const int N = n + (n & 1);
    const JacobiPlan plan = jacobi_plan(m, n);
    const bool beside = plan.launches > 1;  // V's update on the second stream
    if (beside) DH_CHECK_STATUS(dh_aux_stream(h));
    double* A2 = work;
    double2* log = (double2*)(((uintptr_t)(work + (size_t)m * n) + 15) & ~(uintptr_t)15);
    bool pending = false;  // an update of V was queued
    // Sweeps are queued back to back; the flags are read from sweep 6 on
    // (fewer never suffice in FP64 for n > 16), and once a sweep rotates no
    // pair the remaining queued rounds return at once.
    int converged = 0;
    for (int sweep = 0; sweep < kMaxSweeps && !converged; ++sweep) {
        if (plan.own == 0) {
            for (int r = 0; r < N - 1; ++r)
                jacobi_round_kernel<<<N / 2, 64, 0, s>>>(m, n, N, r, A, lda, V, ldv, kJacobiTol,
                                                         words);
            DH_CHECK_LAUNCH();
        } else {
            double2* cs = log + (sweep & 1) * (size_t)(N - 1) * (N / 2);
            double *in = A, *out = plan.launches == 1 ? A : A2;
            int ldi = lda, ldo = plan.launches == 1 ? lda : m;
            for (int k = 0, r = 0; k < plan.launches; ++k) {
                // The rest in equal parts, so every launch has at least one round.
                const int T = dh_cdiv(N - 1 - r, plan.launches - k);
                DH_CHECK_STATUS(
                    launch_rounds(h, m, n, N, r, T, plan.own, in, ldi, out, ldo, cs, words));
                r += T;
                if (plan.launches > 1) {
                    std::swap(in, out);
                    std::swap(ldi, ldo);
                }
            }
        }
        jacobi_sweep_end_kernel<<<1, 64, 0, s>>>(words, sweep);
        DH_CHECK_LAUNCH();
        if (plan.own) {
            // The next sweep reuses the log of the sweep before this one: wait
            // for that one's update of V, then queue this one's.
            if (pending) DH_CHECK_HIP(hipStreamWaitEvent(s, h->ev_update, 0));
            if (beside) {
                DH_CHECK_HIP(hipEventRecord(h->ev_panel, s));
                DH_CHECK_HIP(hipStreamWaitEvent(h->aux, h->ev_panel, 0));
            }
            const int threads = std::min(1024, 64 * dh_cdiv(N / 2 * kJacRows, 64));
            jacobi_apply_kernel<<<dh_cdiv(n, kJacRows), threads, 0, beside ? h->aux : s>>>(
                n, N, log + (sweep & 1) * (size_t)(N - 1) * (N / 2), V, ldv,
                words + 4 + sweep % 4);
            DH_CHECK_LAUNCH();
            if (beside) DH_CHECK_HIP(hipEventRecord(h->ev_update, h->aux));
            pending = beside;
        }
        if (sweep >= 5 || sweep == kMaxSweeps - 1) {
            DH_CHECK_HIP(hipMemcpyAsync(host, words, 3 * sizeof(int), hipMemcpyDeviceToHost, s));
            DH_CHECK_HIP(hipStreamSynchronize(s));
            converged = host[1];
        }
    }
    if (pending) DH_CHECK_HIP(hipStreamWaitEvent(s, h->ev_update, 0));
    *sweeps_out = converged ? host[2] : -1;
    return 0;
}

}  // namespace

extern "C" int dh_gesvj_f64(dh_handle_t h, int m, int n, double* A, int lda, double* sva,
                            double* V, int ldv, int* sweeps) {
    const char* name = "dh_gesvj_f64";
    if (!h) return dh_fail(-1, "%s: NULL handle", name);
    if (m < 0) return dh_fail(-2, "%s: m < 0", name);
    if (n < 0 || n > m) return dh_fail(-3, "%s: need 0 <= n <= m", name);
    if (lda < std::max(1, m)) return dh_fail(-5, "%s: lda < m", name);
    if (ldv < std::max(1, n)) return dh_fail(-8, "%s: ldv < n", name);
    if (sweeps) *sweeps = 0;
    if (n == 0) return 0;
    DH_CHECK_HIP(hipSetDevice(h->device));
    const size_t mn = (size_t)m * n, nn = (size_t)n * n;
    const size_t work = std::max(mn, jacobi_work_doubles(m, n));
    char* ws = (char*)dh_ws(h, DH_WS_EIG, sizeof(double) * (work + nn + n) + sizeof(int) * (n + 64));
    if (!ws) return DH_ERR_ALLOC;
    double* tA = (double*)ws;
    double* tV = tA + work;
    double* key = tV + nn;
    int* ord = (int*)(key + n);
    int* words = ord + n;
    int sw = 0;
    DH_CHECK_STATUS(jacobi_sweeps(h, m, n, A, lda, V, ldv, tA, words, &sw));
    if (sweeps) *sweeps = sw;
    // Singular values = column norms, columns of A and V permuted to descending order.
    column_key_kernel<<<dh_cdiv(n, 4), 256, 0, h->stream>>>(m, n, A, lda, V, ldv, 0, key);
    DH_CHECK_LAUNCH();
    rank_desc_kernel<<<1, 1024, 0, h->stream>>>(n, key, ord);
    DH_CHECK_LAUNCH();
    gather_columns_kernel<<<grid_for(mn), 256, 0, h->stream>>>(m, n, A, lda, ord, key, 0, tA, m,
                                                               sva);
    DH_CHECK_LAUNCH();
    gather_columns_kernel<<<grid_for(nn), 256, 0, h->stream>>>(n, n, V, ldv, ord, key, 0, tV, n,
                                                               nullptr);
    DH_CHECK_LAUNCH();
    copy_cols_kernel<<<grid_for(mn), 256, 0, h->stream>>>(m, n, tA, m, A, lda);
    DH_CHECK_LAUNCH();
    copy_cols_kernel<<<grid_for(nn), 256, 0, h->stream>>>(n, n, tV, n, V, ldv);
    DH_CHECK_LAUNCH();
    DH_CHECK_HIP(hipStreamSynchronize(h->stream));
    if (sw < 0) return dh_fail(1, "%s: no convergence in %d sweeps", name, kMaxSweeps);
    return 0;
}

extern "C" int dh_nystrom_f64(dh_handle_t h, int n, int l, int k, const double* Q, int ldq,
                              const double* W, int ldw, double* Z, int ldz, double* lambda) {
    const char* name = "dh_nystrom_f64";
    if (!h) return dh_fail(-1, "%s: NULL handle", name);
    if (n < 0) return dh_fail(-2, "%s: n < 0", name);
    if (l < 0 || l > n) return dh_fail(-3, "%s: need 0 <= l <= n", name);
    if (k < 0 || k > l) return dh_fail(-4, "%s: need 0 <= k <= l", name);
    if (ldq < std::max(1, n)) return dh_fail(-6, "%s: ldq < n", name);
    if (ldw < std::max(1, n)) return dh_fail(-8, "%s: ldw < n", name);
    if (ldz < std::max(1, n)) return dh_fail(-10, "%s: ldz < n", name);
    if (k == 0 || n == 0) return 0;
    DH_CHECK_HIP(hipSetDevice(h->device));
    const size_t ll = (size_t)l * l;
    char* ws = (char*)dh_ws(h, DH_WS_EIG,
                            sizeof(double) * (2 * ll + (size_t)l * k + l + jacobi_work_doubles(l, l)) +
                                sizeof(int) * (l + 64));
    if (!ws) return DH_ERR_ALLOC;
    double* C = (double*)ws;
    double* V = C + ll;
    double* Vk = V + ll;
    double* lam = Vk + (size_t)l * k;
    double* work = lam + l;
    int* ord = (int*)(work + jacobi_work_doubles(l, l));
    int* words = ord + l;
    // C = Q^T W (testsvm.cpp:126-137), symmetrised.
    DH_CHECK_STATUS(dh_gemm_impl<double>(h, true, false, l, l, n, 1.0, Q, ldq, W, ldw, 0.0, C, l, 0));
    symmetrize_kernel<<<grid_for(ll), 256, 0, h->stream>>>(l, C, l);
    DH_CHECK_LAUNCH();
    int sw = 0;
    DH_CHECK_STATUS(jacobi_sweeps(h, l, l, C, l, V, l, work, words, &sw));
    // C now holds C0 V: lam_j = v_j . (C0 v_j); top k in descending order.
    column_key_kernel<<<dh_cdiv(l, 4), 256, 0, h->stream>>>(l, l, C, l, V, l, 1, lam);
    DH_CHECK_LAUNCH();
    rank_desc_kernel<<<1, 1024, 0, h->stream>>>(l, lam, ord);
    DH_CHECK_LAUNCH();
    // Vk = V[:, top k] diag(sqrt(max(lam, 0))); lambda receives the k eigenvalues.
    gather_columns_kernel<<<grid_for((size_t)l * k), 256, 0, h->stream>>>(l, k, V, l, ord, lam, 1,
                                                                          Vk, l, lambda);
    DH_CHECK_LAUNCH();
    DH_CHECK_STATUS(dh_gemm_impl<double>(h, false, false, n, k, l, 1.0, Q, ldq, Vk, l, 0.0, Z, ldz, 0));
    DH_CHECK_HIP(hipStreamSynchronize(h->stream));
    if (sw < 0) return dh_fail(1, "%s: Jacobi did not converge in %d sweeps", name, kMaxSweeps);
    return 0;
}
