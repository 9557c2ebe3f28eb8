// RBF kernel on gfx950: squared norms, materialised tiles, the fused FP64
// K*Omega projection, and the FP64 error pass.
//
// Reference: rbf_kernel (dkernel.cu:132-190) = vecnorm (102-114) + distance
// GEMM (160-169) + elementwise rbf (116-129), with the K tile copied back to
// the host, replicated, uploaded again and multiplied by Omega in tc_gemm
// (dkernel.h:33-42, dkernel.cu:194-231).  Here the distance GEMM and the
// projection are two MFMA stages of one kernel and K stays in registers.
#include "dh_common.h"
#include "lds_dma.h"
#include "mfma_tile.h"

// ------------------------------------------------------------------ norms

template <typename T>
__global__ __launch_bounds__(256) void sqnorms_kernel(int n, int d, const T* __restrict__ X,
                                                       int ldx, T* __restrict__ nrm) {
    // One wave per point: lanes stride the (contiguous) features, then a
    // butterfly sum.  Summation order differs from the sequential vecnorm.
    int wave = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, lane = threadIdx.x & 63;
    if (wave >= n) return;
    const T* x = X + (size_t)wave * ldx;
    T s = 0;
    for (int f = lane; f < d; f += 64) s += x[f] * x[f];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
    if (lane == 0) nrm[wave] = s;
}

template <typename T>
static int launch_sqnorms(dh_handle_t h, int n, int d, const T* X, int ldx, T* nrm) {
    if (n == 0) return 0;
    sqnorms_kernel<T><<<dh_cdiv(n, 4), 256, 0, h->stream>>>(n, d, X, ldx, nrm);
    DH_CHECK_LAUNCH();
    return 0;
}

extern "C" int dh_sqnorms_f64(dh_handle_t h, int n, int d, const double* X, int ldx,
                              double* nrm) {
    if (!h) return dh_fail(-1, "dh_sqnorms_f64: NULL handle");
    if (n < 0) return dh_fail(-2, "dh_sqnorms_f64: n < 0");
    if (d < 0) return dh_fail(-3, "dh_sqnorms_f64: d < 0");
    if (ldx < max(1, d)) return dh_fail(-5, "dh_sqnorms_f64: ldx < d");
    return launch_sqnorms<double>(h, n, d, X, ldx, nrm);
}

template <typename T>
__device__ __forceinline__ T rbf_exp(T x);
template <>
__device__ __forceinline__ double rbf_exp<double>(double x) {
    return exp(x);
}
template <>
__device__ __forceinline__ float rbf_exp<float>(float x) {
    return __expf(x);  // the reference's fast exp (dkernel.cu:125)
}

// ------------------------------------------------------- materialised tile
//
// Distance GEMM op(A) = Xi^T (point-major, contiguous features), op(B) = Xj,
// then the rbf epilogue on the accumulators: K = yi*yj*exp(-gamma*max(d2, 0)).
template <typename T, int BM, int BN>
__global__ __launch_bounds__(256) void rbf_tile_kernel(int m, int n, int d,
                                                        const T* __restrict__ Xi, int ldxi,
                                                        const T* __restrict__ Xj, int ldxj,
                                                        const T* __restrict__ ni,
                                                        const T* __restrict__ nj,
                                                        const T* __restrict__ yi,
                                                        const T* __restrict__ yj, T gamma,
                                                        T* __restrict__ K, int ldk) {
    constexpr int FM = BM / 32, FN = BN / 32;
    __shared__ T sA[kTileBK][BM + kTilePad];
    __shared__ T sB[kTileBK][BN + kTilePad];
    const int m0 = blockIdx.x * BM, n0 = blockIdx.y * BN;
    typename Mfma<T>::acc_t acc[FM][FN];
    zero_acc<T, FM, FN>(acc);
    tile_mma<T, BM, BN, true, false>(acc, sA, sB, m, n, m0, n0, 0, d, Xi, ldxi, Xj, ldxj);
#pragma unroll
    for (int a = 0; a < FM; ++a)
#pragma unroll
        for (int b = 0; b < FN; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                int i = m0 + tile_row<T, BM, BN>(a, r);
                int j = n0 + tile_col<BM, BN>(b);
                if (i < m && j < n) {
                    T d2 = ni[i] + nj[j] - T(2) * acc[a][b][r];
                    d2 = d2 > T(0) ? d2 : T(0);
                    T v = rbf_exp<T>(-gamma * d2);
                    if (yi) v *= yi[i];
                    if (yj) v *= yj[j];
                    K[i + (size_t)j * ldk] = v;
                }
            }
}

template <typename T>
static int rbf_tile_api(const char* name, dh_handle_t h, int m, int n, int d, const T* Xi,
                        int ldxi, const T* Xj, int ldxj, const T* yi, const T* yj, T gamma, T* K,
                        int ldk) {
    if (!h) return dh_fail(-1, "%s: NULL handle", name);
    if (m < 0) return dh_fail(-2, "%s: m < 0", name);
    if (n < 0) return dh_fail(-3, "%s: n < 0", name);
    if (d < 0) return dh_fail(-4, "%s: d < 0", name);
    if (ldxi < max(1, d)) return dh_fail(-6, "%s: ldxi < d", name);
    if (ldxj < max(1, d)) return dh_fail(-8, "%s: ldxj < d", name);
    if (ldk < max(1, m)) return dh_fail(-13, "%s: ldk < m", name);
    if (m == 0 || n == 0) return 0;
    T* nrm = (T*)dh_ws(h, DH_WS_NORMS, sizeof(T) * ((size_t)m + n));
    if (!nrm) return DH_ERR_ALLOC;
    DH_CHECK_STATUS(launch_sqnorms<T>(h, m, d, Xi, ldxi, nrm));
    DH_CHECK_STATUS(launch_sqnorms<T>(h, n, d, Xj, ldxj, nrm + m));
    dim3 grid(dh_cdiv(m, 64), dh_cdiv(n, 64));
    rbf_tile_kernel<T, 64, 64><<<grid, 256, 0, h->stream>>>(m, n, d, Xi, ldxi, Xj, ldxj, nrm,
                                                             nrm + m, yi, yj, gamma, K, ldk);
    DH_CHECK_LAUNCH();
    return 0;
}

extern "C" int dh_rbf_tile_f64(dh_handle_t h, int m, int n, int d, const double* Xi, int ldxi,
                               const double* Xj, int ldxj, const double* yi, const double* yj,
                               double gamma, double* K, int ldk) {
    return rbf_tile_api<double>("dh_rbf_tile_f64", h, m, n, d, Xi, ldxi, Xj, ldxj, yi, yj, gamma,
                                K, ldk);
}
extern "C" int dh_rbf_tile_f32(dh_handle_t h, int m, int n, int d, const float* Xi, int ldxi,
                               const float* Xj, int ldxj, const float* yi, const float* yj,
                               float gamma, float* K, int ldk) {
    return rbf_tile_api<float>("dh_rbf_tile_f32", h, m, n, d, Xi, ldxi, Xj, ldxj, yi, yj, gamma, K,
                               ldk);
}

// ------------------------------------------------- fused FP64 K * Omega
//
// Workgroup: 4 waves, 64 rows i (16 per wave).  The j loop walks Xj and
// Omega in chunks of 16 points staged in LDS.  Per chunk each wave
//   1. forms S^T = Xj_chunk * Xi_wave^T (16 j x 16 i) with DK f64 MFMAs in two
//      independent accumulation chains.  Feature f = g*DK + kk is k-slot g of
//      MFMA kk, so lane (g, li) reads its A operands (point li of the chunk)
//      as consecutive doubles of a point-major LDS row, two per 16-byte read,
//      and keeps its B operands (row li of Xi, features g*DK ..) in registers;
//   2. turns its 4 accumulators into K values in place (exp epilogue);
//   3. uses them directly as the A operand of the projection MFMAs: lane L
//      holds S^T[L/16+4r][L%16] = K[i=L%16][j=4r+L/16] (f64 accumulator
//      layout), i.e. MFMA r contracts over j = 4r..4r+3; Omega is staged in
//      LDS so that lane L reads the B operands of MFMAs 2h and 2h+1 of block
//      cb as one 16-byte pair sO[cb][h][L ^ 4(L/16)] = (Omega[j0+4(2h)+L/16][c],
//      Omega[j0+4(2h+1)+L/16][c]), c = c0 + 16cb + L%16.  The XOR keeps each
//      aligned group of 8 lanes on 8 consecutive pairs (conflict-free reads)
//      and spreads the staging stores, whose 64 lanes cover 4 columns x 16
//      points, over all banks (2 cycles per store instead of 8).
// The chunks go through two LDS buffers: the global loads of chunk t+1 are
// issued into registers before chunk t is computed and stored to the other
// buffer after it, so one barrier per chunk orders both.  (With one buffer,
// single 8-byte operand reads consumed at once and the accumulators moved
// between register files every chunk, the pass ran at 38% of the FP64 MFMA
// peak; this layout runs at 51%.)
// Labels are folded: yj scales Omega as it is staged, yi scales the output.
// The projection accumulators (NCB blocks of 16 columns) stay in registers
// for the whole j loop; Y is written once.
// exp(x) without branches for the kernel's exponents x = -gamma d2 <= 0
// (valid up to x = 709): k = rint(x log2 e); r = (x - k LN2_HI) - k LN2_LO, a
// Cody-Waite reduction with LN2_HI = ln 2 rounded to 32 significant bits (k
// LN2_HI exact for |k| < 2^21) and LN2_LO = ln 2 - LN2_HI rounded to double;
// e^r by its Taylor series to degree 13 in Horner form (truncation below
// 2^-55 for |r| <= ln2 / 2); then 2^k by ldexp, which rounds subnormal
// results and gives 0 below 2^-1075.  Within 1 ulp of libm's exp over
// [-746, 0] (an exact-FMA emulation checked on 20000 points and the edges).
__device__ __forceinline__ double exp_kernel_f64(double x) {
    x = fmax(x, -746.0);
    const double k = rint(x * 1.4426950408889634);
    double r = fma(-k, 0x1.62e42ff000000p-1, x);
    r = fma(-k, -0x1.718432a1b0e26p-35, r);
    double p = 1.6059043836821613e-10;  // 1/13!
    p = fma(p, r, 2.08767569878681e-09);
    p = fma(p, r, 2.505210838544172e-08);
    p = fma(p, r, 2.755731922398589e-07);
    p = fma(p, r, 2.7557319223985893e-06);
    p = fma(p, r, 2.48015873015873e-05);
    p = fma(p, r, 1.984126984126984e-04);
    p = fma(p, r, 1.388888888888889e-03);
    p = fma(p, r, 8.333333333333333e-03);
    p = fma(p, r, 4.1666666666666664e-02);
    p = fma(p, r, 1.6666666666666666e-01);
    p = fma(p, r, 0.5);
    p = fma(p, r, 1.0);
    p = fma(p, r, 1.0);
    return ldexp(p, (int)k);
}

typedef double d2v __attribute__((ext_vector_type(2)));

// Omega (or Q) with the labels folded in, in the kernel's LDS image: for
// 16-point chunk t, column block cb (of ncbp) and h, the 64 pairs
// Opk[((t ncbp + cb) 2 + h) 64 + (L ^ 4(L/16))] = (y_j O[j][c], y_{j+4} O[j+4][c]),
// j = 16t + 8h + L/16, c = 16cb + L%16, zero outside n x l; one thread per pair.
__global__ __launch_bounds__(256) void pack_omega_f64_kernel(int n, int l, int nch, int ncbp,
                                                             const double* __restrict__ O,
                                                             int ldo,
                                                             const double* __restrict__ yj,
                                                             d2v* __restrict__ Opk) {
    const long idx = (long)blockIdx.x * 256 + threadIdx.x;
    if (idx >= (long)nch * ncbp * 128) return;
    const int s = (int)(idx & 63), h = (int)((idx >> 6) & 1);
    const long tc = idx >> 7;
    const int cb = (int)(tc % ncbp), t = (int)(tc / ncbp);
    const int L = s ^ ((s >> 4) << 2);
    const int j = 16 * t + 8 * h + (L >> 4), c = 16 * cb + (L & 15);
    d2v v = {0.0, 0.0};
    if (c < l) {
        if (j < n) v[0] = O[j + (size_t)c * ldo] * (yj ? yj[j] : 1.0);
        if (j + 4 < n) v[1] = O[j + 4 + (size_t)c * ldo] * (yj ? yj[j + 4] : 1.0);
    }
    Opk[idx] = v;
}

template <int DK, int NCB, bool PK>
__global__ __launch_bounds__(256) void rbf_project_f64_kernel(
    int m, int n, int d, int l, const double* __restrict__ Xi, int ldxi,
    const double* __restrict__ Xj, int ldxj, const double* __restrict__ ni,
    const double* __restrict__ nj, const double* __restrict__ yi, const double* __restrict__ yj,
    double gamma, const double* __restrict__ O, int ldo, const d2v* __restrict__ Opk, int ncbp,
    double beta, double* __restrict__ Y, int ldy, int jps, long ystride) {
    constexpr int JB = 16;
    {  // split z of the j range: points [z jps, min((z + 1) jps, n)), partial into Y + z ystride
        const int j0 = blockIdx.z * jps;
        n = min(jps, n - j0);
        Xj += (size_t)j0 * ldxj;
        nj += j0;
        if (yj) yj += j0;
        O += j0;
        if (PK) Opk += (size_t)(j0 / JB) * ncbp * 128;
        Y += blockIdx.z * ystride;
    }
    constexpr int FD = DK * 4;  // padded feature count
    constexpr int XP = FD + 2;  // LDS pitch of a point (odd multiple of 16 bytes: no conflicts)
    __shared__ double sX[2][JB * XP];
    __shared__ d2v sO[2][NCB][2][64];
    __shared__ double sN[2][JB];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 4, li = lane & 15;
    const int c0 = blockIdx.y * NCB * 16;
    const int rbase = blockIdx.x * 64 + wave * 16;
    const int row = rbase + li;

    double xr[DK];
#pragma unroll
    for (int kk = 0; kk < DK; ++kk) {
        const int f = g * DK + kk;
        xr[kk] = (row < m && f < d) ? Xi[f + (size_t)row * ldxi] : 0.0;
    }
    const double nrow = (row < m) ? ni[row] : 0.0;
    dh_d4 acc[NCB];
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) acc[cb] = dh_d4{0, 0, 0, 0};

    // Staging of a chunk: every load is issued before any LDS store, from
    // addresses clamped into the operands (a load under a branch gets a wait
    // of its own).  Thread tid always stages point jj = tid % JB of the Omega
    // block, so its label is one load per chunk.
    constexpr int NXL = JB * FD / 256, NOL = JB * NCB * 16 / 256;
    static_assert(JB * FD % 256 == 0 && JB * NCB * 16 % 256 == 0, "staging split");
    double px[NXL], po[PK ? 1 : NOL], pn, yv;
    // PK: the chunk's packed Omega image (NCB x 2 KB, contiguous) goes to LDS
    // by direct copies, 1 KB per wave instruction.
    auto dma_omega = [&](int j0, int b) {
        const d2v* src = Opk + ((size_t)(j0 / JB) * ncbp + blockIdx.y * NCB) * 128;
#pragma unroll
        for (int k = 0; k < 2 * NCB; k += 4) {
            const int kk = k + wave;
            if ((2 * NCB) % 4 == 0 || kk < 2 * NCB)
                dma16(src + kk * 64, (unsigned)lane * 16u, &sO[b][kk >> 1][kk & 1][0]);
        }
    };
    auto load = [&](int j0) {
#pragma unroll
        for (int u = 0; u < NXL; ++u) {
            const int e = tid + 256 * u, jj = e / FD, f = e % FD;
            px[u] = Xj[min(f, d - 1) + (size_t)min(j0 + jj, n - 1) * ldxj];
        }
        const int jo = j0 + (tid % JB);
        if constexpr (!PK) {
            yv = yj ? yj[min(jo, n - 1)] : 1.0;
#pragma unroll
            for (int u = 0; u < NOL; ++u) {
                const int e = tid + 256 * u, cl = e / JB;
                po[u] = O[min(jo, n - 1) + (size_t)min(c0 + cl, l - 1) * ldo];
            }
        }
        pn = nj[min(j0 + (tid % JB), n - 1)];
    };
    auto store = [&](int j0, int b) {
        const int jo = j0 + (tid % JB);
#pragma unroll
        for (int u = 0; u < NXL; ++u) {
            const int e = tid + 256 * u, jj = e / FD, f = e % FD;
            sX[b][jj * XP + f] = (j0 + jj < n && f < d) ? px[u] : 0.0;
        }
        double* so = (double*)&sO[b][0][0][0];
#pragma unroll
        for (int u = 0; u < (PK ? 0 : NOL); ++u) {
            const int e = tid + 256 * u, jj = e % JB, cl = e / JB;
            const int r = jj >> 2, ln = (jj & 3) * 16 + ((cl & 15) ^ ((jj & 3) << 2));
            so[(((cl >> 4) * 2 + (r >> 1)) * 64 + ln) * 2 + (r & 1)] =
                (jo < n && c0 + cl < l) ? po[u] * yv : 0.0;
        }
        if (tid < JB) sN[b][tid] = (j0 + tid < n) ? pn : 0.0;
    };

    load(0);
    if constexpr (PK) dma_omega(0, 0);
    store(0, 0);
    if constexpr (PK) wait_vm();
    __syncthreads();
    int b = 0;
    for (int j0 = 0; j0 < n; j0 += JB) {
        const bool more = j0 + JB < n;  // uniform
        if (more) {
            load(j0 + JB);
            if constexpr (PK) dma_omega(j0 + JB, b ^ 1);
        }
        dh_d4 s0 = dh_d4{0, 0, 0, 0}, s1 = dh_d4{0, 0, 0, 0};
        const double* xrow = &sX[b][li * XP + g * DK];
#pragma unroll
        for (int kk = 0; kk < DK; kk += 2) {
            const d2v a2 = *(const d2v*)(xrow + kk);
            s0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a2[0], xr[kk], s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a2[1], xr[kk + 1], s1, 0, 0, 0);
        }
        double kv[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            double d2 = nrow + sN[b][g + 4 * r] - 2.0 * (s0[r] + s1[r]);
            d2 = d2 > 0.0 ? d2 : 0.0;
            kv[r] = exp_kernel_f64(-gamma * d2);
        }
        const int sl = lane ^ ((lane >> 4) << 2);
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb) {
            const d2v o01 = sO[b][cb][0][sl], o23 = sO[b][cb][1][sl];
            acc[cb] = __builtin_amdgcn_mfma_f64_16x16x4f64(kv[0], o01[0], acc[cb], 0, 0, 0);
            acc[cb] = __builtin_amdgcn_mfma_f64_16x16x4f64(kv[1], o01[1], acc[cb], 0, 0, 0);
            acc[cb] = __builtin_amdgcn_mfma_f64_16x16x4f64(kv[2], o23[0], acc[cb], 0, 0, 0);
            acc[cb] = __builtin_amdgcn_mfma_f64_16x16x4f64(kv[3], o23[1], acc[cb], 0, 0, 0);
        }
        if (more) store(j0 + JB, b ^ 1);
        if constexpr (PK) wait_vm();
        __syncthreads();
        b ^= 1;
    }
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            int i = rbase + g + 4 * r, c = c0 + 16 * cb + li;
            if (i < m && c < l) {
                double v = acc[cb][r];
                if (yi) v *= yi[i];
                double* yp = Y + i + (size_t)c * ldy;
                *yp = (beta == 0.0) ? v : v + beta * (*yp);
            }
        }
}

// The kept layout: K without labels as the projection MFMAs take it, 128 pairs
// per (16-point chunk, 16-row block), pair h 64 + L = (kv[2h], kv[2h + 1]) of
// lane L with kv as in rbf_project_f64_kernel; nrb row blocks per chunk.  Chunks
// are outermost because all waves walk them together: the reads and writes of
// any moment lie side by side.

// Stores block (row block rb, chunk t) of K in the kept layout and, with
// `mirror`, the transposed block (t, rb) through the wave's 16 x 17 of LDS.
__device__ __forceinline__ void store_kept(double (&kv)[4], int rb, int t, int nch, int nrb,
                                           bool mirror, double (*sT)[17], d2v* __restrict__ Kk) {
    const int lane = threadIdx.x & 63, g = lane >> 4, li = lane & 15;
    if (t < nch) {  // row blocks are padded to whole tiles, chunks are not
        d2v* kp = Kk + ((size_t)t * nrb + rb) * 128 + lane;
        kp[0] = d2v{kv[0], kv[1]};
        kp[64] = d2v{kv[2], kv[3]};
    }
    if (!mirror) return;
#pragma unroll
    for (int r = 0; r < 4; ++r) sT[4 * r + g][li] = kv[r];
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int r = 0; r < 4; ++r) kv[r] = sT[li][4 * r + g];
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (rb < nch) {
        d2v* kp = Kk + ((size_t)rb * nrb + t) * 128 + lane;
        kp[0] = d2v{kv[0], kv[1]};
        kp[64] = d2v{kv[2], kv[3]};
    }
}

// K of one point set with up to 4 DK features, in the kept layout and with the
// fused kernel's bits: its distance stage (products, exp) on one triangle of
// 64 x 64 tiles, whose strict part is stored a second time transposed; products
// and norms commute.  Workgroup (bi, z): 64 rows, the part of points [64 z seg,
// 64 (z + 1) seg) from row tile bi on.  n = 65536, d = 128: 14.2 ms, 39 TFLOP/s beside
// 34 GB of writes (a fused pass that stores K as it goes takes 29.5 ms more than
// a kept one); n = 8192, d = 64: 0.166 ms against 0.31.
template <int DK>
__global__ __launch_bounds__(256) void form_sym_f64_kernel(int n, int d,
                                                           const double* __restrict__ X, int ldx,
                                                           const double* __restrict__ nrm,
                                                           double gamma, int seg,
                                                           d2v* __restrict__ Kk, int nrb) {
    constexpr int JB = 16, FD = DK * 4, XP = FD + 2;
    __shared__ double sX[2][JB * XP];
    __shared__ double sN[2][JB];
    __shared__ double sT[4][16][17];
    const int bi = blockIdx.x, nt = gridDim.x;
    const int tb = max((int)blockIdx.y * seg, bi), te = min(((int)blockIdx.y + 1) * seg, nt);
    if (tb >= te) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, li = lane & 15;
    const int rb = 4 * bi + wave, row = 16 * rb + li, nch = (n + JB - 1) / JB;
    double xr[DK];
#pragma unroll
    for (int kk = 0; kk < DK; ++kk) {
        const int f = g * DK + kk;
        xr[kk] = (row < n && f < d) ? X[f + (size_t)row * ldx] : 0.0;
    }
    const double nrow = (row < n) ? nrm[row] : 0.0;
    constexpr int NXL = JB * FD / 256;
    double px[NXL], pn;
    auto load = [&](int j0) {
#pragma unroll
        for (int u = 0; u < NXL; ++u) {
            const int e = tid + 256 * u, jj = e / FD, f = e % FD;
            px[u] = X[min(f, d - 1) + (size_t)min(j0 + jj, n - 1) * ldx];
        }
        pn = nrm[min(j0 + (tid % JB), n - 1)];
    };
    auto store = [&](int j0, int b) {
#pragma unroll
        for (int u = 0; u < NXL; ++u) {
            const int e = tid + 256 * u, jj = e / FD, f = e % FD;
            sX[b][jj * XP + f] = (j0 + jj < n && f < d) ? px[u] : 0.0;
        }
        if (tid < JB) sN[b][tid] = (j0 + tid < n) ? pn : 0.0;
    };
    load(64 * tb);
    store(64 * tb, 0);
    __syncthreads();
    int b = 0;
    for (int t = 4 * tb; t < 4 * te; ++t) {
        const bool more = t + 1 < 4 * te;  // uniform
        if (more) load(JB * (t + 1));
        dh_d4 s0 = dh_d4{0, 0, 0, 0}, s1 = dh_d4{0, 0, 0, 0};
        const double* xrow = &sX[b][li * XP + g * DK];
#pragma unroll
        for (int kk = 0; kk < DK; kk += 2) {
            const d2v a2 = *(const d2v*)(xrow + kk);
            s0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a2[0], xr[kk], s0, 0, 0, 0);
            s1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a2[1], xr[kk + 1], s1, 0, 0, 0);
        }
        double kv[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            double d2 = nrow + sN[b][g + 4 * r] - 2.0 * (s0[r] + s1[r]);
            d2 = d2 > 0.0 ? d2 : 0.0;
            kv[r] = exp_kernel_f64(-gamma * d2);
        }
        store_kept(kv, rb, t, nch, nrb, (t >> 2) != bi, sT[wave], Kk);
        if (more) store(JB * (t + 1), b ^ 1);
        __syncthreads();
        b ^= 1;
    }
}

// K without labels in the kept layout, for points of any number of features: 64
// x 64 distance tiles (tile_mma) with the points of the columns as tile rows, so
// that the accumulators of lane (g, li) are already its pairs.  SYM (Xi = Xj): one
// triangle of tiles, of which the strict part is stored a second time with every
// 16 x 16 block transposed through LDS; the products and norms commute, so both
// halves have the bits of their own tile.
template <bool SYM>
__global__ __launch_bounds__(256) void form_f64_kernel(int m, int n, int d,
                                                       const double* __restrict__ Xi, int ldxi,
                                                       const double* __restrict__ Xj, int ldxj,
                                                       const double* __restrict__ ni,
                                                       const double* __restrict__ nj,
                                                       double gamma, d2v* __restrict__ Kk,
                                                       int nrb) {
    __shared__ double sA[kTileBK][64 + kTilePad];
    __shared__ double sB[kTileBK][64 + kTilePad];
    __shared__ double sT[4][16][17];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, li = lane & 15;
    int bj = blockIdx.x, bi = blockIdx.y;  // tile rows: points of Xj; tile columns: of Xi
    if (SYM) {
        const int t = blockIdx.x;
        bi = (int)((sqrtf(8.0f * (float)t + 1.0f) - 1.0f) * 0.5f);
        while ((bi + 1) * (bi + 2) / 2 <= t) ++bi;
        while (bi * (bi + 1) / 2 > t) --bi;
        bj = t - bi * (bi + 1) / 2;
    }
    dh_d4 acc[2][2];
    zero_acc<double, 2, 2>(acc);
    tile_mma<double, 64, 64, true, false>(acc, sA, sB, n, m, 64 * bj, 64 * bi, 0, d, Xj, ldxj, Xi,
                                          ldxi);
    const int nch = (n + 15) / 16;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const int t = 4 * bj + (wave & 1) * 2 + a, rb = 4 * bi + (wave >> 1) * 2 + b;
            const double nrow = ni[min(16 * rb + li, m - 1)];
            double kv[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = 16 * rb + li, j = 16 * t + 4 * r + g;
                double d2 = nrow + nj[min(j, n - 1)] - 2.0 * acc[a][b][r];
                // Past the last point 1, which a negative gamma cannot take to infinity.
                d2 = d2 > 0.0 && i < m && j < n ? d2 : 0.0;
                kv[r] = exp(-gamma * d2);
            }
            store_kept(kv, rb, t, nch, nrb, SYM && bi != bj, sT[wave], Kk);
        }
}

// Y = K O from K values in the kept layout, with the packed Omega image, chunk
// order and MFMAs of the fused kernel, so it returns that kernel's bits where
// the values are its values.  Rows, columns and splits as there; what is gone is the
// distance product (2d of the 2(d + l) flops per entry), the exp, and the
// staging of X, and with it the registers and LDS that held the fused kernel
// to one workgroup per CU at l = 272: here two fit.  K comes from HBM once per
// column group, 8 bytes per entry, a chunk ahead in registers.
template <int NCB>
__global__ __launch_bounds__(256, 2) void kept_project_f64_kernel(
    int m, int n, int l, const d2v* __restrict__ Kk, int nrb, const double* __restrict__ yi,
    const d2v* __restrict__ Opk, int ncbp, double* __restrict__ Y, int ldy, int jps,
    long ystride) {
    constexpr int JB = 16;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int jz = blockIdx.z * jps;
    const int nch = (min(jps, n - jz) + JB - 1) / JB;
    Opk += ((size_t)(jz / JB) * ncbp + blockIdx.y * NCB) * 128;
    Kk += ((size_t)(jz / JB) * nrb + blockIdx.x * 4 + wave) * 128 + lane;
    const size_t kstep = (size_t)nrb * 128;
    Y += blockIdx.z * ystride;
    __shared__ d2v sO[2][NCB][2][64];
    const int g = lane >> 4, li = lane & 15, sl = lane ^ (g << 2);
    dh_d4 acc[NCB];
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb) acc[cb] = dh_d4{0, 0, 0, 0};
    auto dma_omega = [&](int t, int b) {
        const d2v* src = Opk + (size_t)t * ncbp * 128;
#pragma unroll
        for (int k = 0; k < 2 * NCB; k += 4) {
            const int kk = k + wave;
            if ((2 * NCB) % 4 == 0 || kk < 2 * NCB)
                dma16(src + kk * 64, (unsigned)lane * 16u, &sO[b][kk >> 1][kk & 1][0]);
        }
    };
    d2v k01 = Kk[0], k23 = Kk[64];
    dma_omega(0, 0);
    wait_vm();
    __syncthreads();
    for (int t = 0; t < nch; ++t) {
        const int b = t & 1, tn = min(t + 1, nch - 1);
        const d2v n01 = Kk[tn * kstep], n23 = Kk[tn * kstep + 64];
        if (t + 1 < nch) dma_omega(t + 1, b ^ 1);
#pragma unroll
        for (int cb = 0; cb < NCB; ++cb) {
            const d2v o01 = sO[b][cb][0][sl], o23 = sO[b][cb][1][sl];
            acc[cb] = __builtin_amdgcn_mfma_f64_16x16x4f64(k01[0], o01[0], acc[cb], 0, 0, 0);
            acc[cb] = __builtin_amdgcn_mfma_f64_16x16x4f64(k01[1], o01[1], acc[cb], 0, 0, 0);
            acc[cb] = __builtin_amdgcn_mfma_f64_16x16x4f64(k23[0], o23[0], acc[cb], 0, 0, 0);
            acc[cb] = __builtin_amdgcn_mfma_f64_16x16x4f64(k23[1], o23[1], acc[cb], 0, 0, 0);
        }
        k01 = n01;
        k23 = n23;
        wait_vm();
        __syncthreads();
    }
#pragma unroll
    for (int cb = 0; cb < NCB; ++cb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int i = blockIdx.x * 64 + wave * 16 + g + 4 * r;
            const int c = (blockIdx.y * NCB + cb) * 16 + li;
            if (i < m && c < l) {
                double v = acc[cb][r];
                if (yi) v *= yi[i];
                Y[i + (size_t)c * ldy] = v;
            }
        }
}

template <int DK, int NCB>
static void launch_project_f64(dh_handle_t h, dim3 grid, int m, int n, int d, int l,
                               const double* Xi, int ldxi, const double* Xj, int ldxj,
                               const double* ni, const double* nj, const double* yi,
                               const double* yj, double gamma, const double* O, int ldo,
                               const d2v* Opk, int ncbp, double beta, double* Y, int ldy, int jps,
                               long ystride) {
    if constexpr (DK < 64 || NCB <= 12) {  // d > 128 with 17 blocks is never selected (spills)
        dh_timing_begin(h);
        if (Opk)
            rbf_project_f64_kernel<DK, NCB, true><<<grid, 256, 0, h->stream>>>(
                m, n, d, l, Xi, ldxi, Xj, ldxj, ni, nj, yi, yj, gamma, O, ldo, Opk, ncbp, beta, Y,
                ldy, jps, ystride);
        else
            rbf_project_f64_kernel<DK, NCB, false><<<grid, 256, 0, h->stream>>>(
                m, n, d, l, Xi, ldxi, Xj, ldxj, ni, nj, yi, yj, gamma, O, ldo, nullptr, 0, beta, Y,
                ldy, jps, ystride);
        dh_timing_end(h);
    }
}

template <int DK>
static int dispatch_ncb(dh_handle_t h, int ncb, dim3 grid, int m, int n, int d, int l,
                        const double* Xi, int ldxi, const double* Xj, int ldxj, const double* ni,
                        const double* nj, const double* yi, const double* yj, double gamma,
                        const double* O, int ldo, const d2v* Opk, int ncbp, double beta,
                        double* Y, int ldy, int jps, long ystride) {
#define DH_NCB(N)                                                                              \
    case N:                                                                                    \
        launch_project_f64<DK, N>(h, grid, m, n, d, l, Xi, ldxi, Xj, ldxj, ni, nj, yi, yj, gamma, \
                                  O, ldo, Opk, ncbp, beta, Y, ldy, jps, ystride);              \
        break;
    switch (ncb) {
        DH_NCB(1)
        DH_NCB(2)
        DH_NCB(3)
        DH_NCB(4)
        DH_NCB(5)
        DH_NCB(6)
        DH_NCB(8)
        DH_NCB(9)
        DH_NCB(12)
        DH_NCB(17)
        default:
            return dh_fail(DH_ERR_UNSUPPORTED, "rbf_project_f64: no kernel for %d column blocks",
                           ncb);
    }
#undef DH_NCB
    DH_CHECK_LAUNCH();
    return 0;
}

// Smallest instantiated column-block count >= want.
static int ncb_instance(int want) {
    static const int inst[] = {1, 2, 3, 4, 5, 6, 8, 9, 12, 17};
    for (int v : inst)
        if (v >= want) return v;
    return 17;
}

// Omega (labels folded in) as the fused kernels' LDS images, ncbp column blocks.
static int pack_omega_f64(dh_handle_t h, int n, int l, int ncbp, const double* O, int ldo,
                          const double* yj, const d2v** Opk) {
    const int nch = dh_cdiv(n, 16);
    const long pairs = (long)nch * ncbp * 128;
    d2v* P = (d2v*)dh_ws(h, DH_WS_PACK64, sizeof(d2v) * (size_t)pairs);
    if (!P) return DH_ERR_ALLOC;
    pack_omega_f64_kernel<<<dh_cdiv(pairs, 256), 256, 0, h->stream>>>(n, l, nch, ncbp, O, ldo, yj,
                                                                     P);
    DH_CHECK_LAUNCH();
    *Opk = P;
    return 0;
}

// Column blocking of a pass on kept K values: without the distance operands 17
// column blocks fit at every d, and how the columns are grouped changes no bit.
static void kept_columns(int l, int* ncb, int* groups) {
    const int ncb_total = dh_cdiv(l, 16);
    *ncb = ncb_instance(dh_cdiv(ncb_total, dh_cdiv(ncb_total, 17)));
    *groups = dh_cdiv(ncb_total, *ncb);
}

// Y (m x l) = K O from K values in the kept layout (nrb row blocks per chunk),
// Omega packed in ncb x groups column blocks.
static int launch_kept_f64(dh_handle_t h, int m, int n, int l, int ncb, int groups,
                           const double* yi, const d2v* Opk, double* Y, int ldy, int jps,
                           int splits, long ystride, const void* keep, int nrb) {
    dim3 grid(dh_cdiv(m, 64), groups, splits);
#define DH_NCB(N)                                                                         \
    case N:                                                                               \
        kept_project_f64_kernel<N><<<grid, 256, 0, h->stream>>>(                          \
            m, n, l, (const d2v*)keep, nrb, yi, Opk, groups* ncb, Y, ldy, jps, ystride);  \
        break;
    switch (ncb) {
        DH_NCB(1)
        DH_NCB(2)
        DH_NCB(3)
        DH_NCB(4)
        DH_NCB(5)
        DH_NCB(6)
        DH_NCB(8)
        DH_NCB(9)
        DH_NCB(12)
        default:
            DH_NCB(17)
    }
#undef DH_NCB
    DH_CHECK_LAUNCH();
    return 0;
}

static int project_f64_kept(dh_handle_t h, int m, int n, int l, const double* yi,
                            const double* yj, const double* O, int ldo, double* Y, int ldy,
                            int jps, int splits, long ystride, const void* keep) {
    int ncb, groups;
    kept_columns(l, &ncb, &groups);
    const d2v* Opk = nullptr;
    DH_CHECK_STATUS(pack_omega_f64(h, n, l, groups * ncb, O, ldo, yj, &Opk));
    dh_timing_begin(h);
    DH_CHECK_STATUS(launch_kept_f64(h, m, n, l, ncb, groups, yi, Opk, Y, ldy, jps, splits, ystride,
                                    keep, 4 * dh_cdiv(m, 64)));
    dh_timing_end(h);
    return 0;
}

// Y = beta Y + sum over the splits z (in order) of P[z ystride + i + c m].
__global__ __launch_bounds__(256) void sum_splits_f64_kernel(int m, int l, int splits,
                                                             const double* __restrict__ P,
                                                             long ystride, double beta,
                                                             double* __restrict__ Y, int ldy) {
    const long e = (long)blockIdx.x * 256 + threadIdx.x;
    if (e >= (long)m * l) return;
    const int i = (int)(e % m), c = (int)(e / m);
    double v = 0.0;
    for (int z = 0; z < splits; ++z) v += P[z * ystride + e];
    double* yp = Y + i + (size_t)c * ldy;
    *yp = (beta == 0.0) ? v : v + beta * (*yp);
}

// Bytes of K (m x n) in the kept layout: whole 64-row tiles, 16-point chunks.
static size_t kept_bytes(int m, int n) {
    return sizeof(double) * ((size_t)dh_cdiv(m, 64) * 64) * ((size_t)dh_cdiv(n, 16) * 16);
}

// Rows per block of K (m x n): equal blocks of at most 2^27 entries as laid out,
// with the columns padded to whole chunks, and of at most 65535 row tiles, which
// lie in the y dimension of form_f64_kernel's grid (its customary limit, reached
// with n <= 31; ROCm 7.2 launched 65538 all the same).
static int block_rows(int m, int n) {
    const long fit = (1L << 27) / ((n + 15L) / 16 * 16) / 64 * 64;
    const int most = (int)std::min(64L * 65535, std::max(64L, fit));
    return dh_cdiv(dh_cdiv(m, dh_cdiv(m, most)), 64) * 64;
}

// Above 256 features a wave's rows of Xi no longer fit in registers.  K is then
// formed in the kept layout by distance tiles, in row blocks of at most 2^27
// entries (1 GiB), and each block multiplied into Omega by
// kept_project_f64_kernel.  The same split as rbf_kernel's explicit tiles
// (dkernel.cu:144-178).  With `keep` K is one block there: kmode 1 forms it,
// from one triangle where both point sets are the same; kmode 2 takes it as an
// earlier pass left it.  The j range is split until a row block has two
// workgroups per CU, into parts of at least four chunks of 32 points (2000 x 2000, d =
// 300, l = 272: 145 us, with parts of 16 chunks 255, through the GEMM 155), also where
// K is kept, so that both return the same bits.
// (Column-major blocks through the 64 x 64 GEMM: n = 9000, d = 600, l = 74 took
// 2.13 + 0.49 ms per pass; forming one triangle takes 1.07 and a pass 0.33.
// One pass over row blocks, d = 300, l = 74, GEMM -> here, and with the split
// chosen from all m rows: n = 40000 30.2 -> 26.0 and 57.8 ms, n = 65536 76.9 -> 69.8
// and 203 ms, 300 x 500000 3.8 -> 3.4 and 11.5 ms.  With K kept the splits cost
// 1% at n = 65536, l = 272 and gain 14% at n = 40000.)  The partial products take at
// most 1 GiB, or 4 GiB beside a kept K, in parts of the rows.
static int project_f64_blocked(dh_handle_t h, int m, int n, int d, int l, const double* Xi,
                               int ldxi, const double* Xj, int ldxj, const double* ni,
                               const double* nj, const double* yi, const double* yj, double gamma,
                               const double* O, int ldo, double beta, double* Y, int ldy,
                               void* keep, int kmode) {
    if (n == 0)  // K has no columns: Y = beta Y
        return dh_gemm_impl<double>(h, false, false, m, l, 0, 1.0, O, 1, O, ldo, beta, Y, ldy, 0);
    const int rows = std::min(m, block_rows(m, n)), mb = keep ? m : rows;
    void* Kb = keep ? keep : dh_ws(h, DH_WS_KBLOCK, kept_bytes(mb, n));
    if (!Kb) return DH_ERR_ALLOC;
    int ncb, groups;
    kept_columns(l, &ncb, &groups);
    const int nch = dh_cdiv(n, 32);
    int splits = 1;
    while ((long)dh_cdiv(rows, 64) * groups * splits < 2L * h->num_cu && nch >= 8 * splits)
        splits *= 2;
    const int jps = splits == 1 ? n : dh_cdiv(nch, splits) * 32;
    splits = dh_cdiv(n, jps);
    const bool direct = splits == 1 && beta == 0.0;
    double* P = nullptr;
    int pr = mb;  // rows per launch
    if (!direct) {
        const long fit = (keep ? 1L << 29 : 1L << 27) / ((long)l * splits) / 64 * 64;
        pr = (int)std::min<long>(mb, std::max(64L, fit));
        P = (double*)dh_ws(h, DH_WS_SPLITN, sizeof(double) * (size_t)pr * l * splits);
        if (!P) return DH_ERR_ALLOC;
    }
    const d2v* Opk = nullptr;
    DH_CHECK_STATUS(pack_omega_f64(h, n, l, groups * ncb, O, ldo, yj, &Opk));
    const bool sym = keep && Xi == Xj && ldxi == ldxj && m == n && ni == nj;
    dh_timing_begin(h);
    for (int i0 = 0; i0 < m; i0 += mb) {
        const int ib = std::min(mb, m - i0), bt = dh_cdiv(ib, 64), jt = dh_cdiv(n, 64);
        if (kmode != 2) {
            if (sym)
                form_f64_kernel<true><<<(unsigned)((long)bt * (bt + 1) / 2), 256, 0, h->stream>>>(
                    ib, n, d, Xi, ldxi, Xj, ldxj, ni, nj, gamma, (d2v*)Kb, 4 * bt);
            else
                form_f64_kernel<false><<<dim3(jt, bt), 256, 0, h->stream>>>(
                    ib, n, d, Xi + (size_t)i0 * ldxi, ldxi, Xj, ldxj, ni + i0, nj, gamma,
                    (d2v*)Kb, 4 * bt);
            DH_CHECK_LAUNCH();
        }
        for (int r0 = 0; r0 < ib; r0 += pr) {
            const int rb = std::min(pr, ib - r0);
            double* y0 = Y + i0 + r0;
            const long ystride = (long)rb * l;
            DH_CHECK_STATUS(launch_kept_f64(h, rb, n, l, ncb, groups, yi ? yi + i0 + r0 : nullptr,
                                            Opk, direct ? y0 : P, direct ? ldy : rb, jps, splits,
                                            ystride, (const d2v*)Kb + (size_t)(r0 / 16) * 128,
                                            4 * bt));
            if (direct) continue;
            sum_splits_f64_kernel<<<dh_cdiv(ystride, 256), 256, 0, h->stream>>>(
                rb, l, splits, P, ystride, beta, y0, ldy);
            DH_CHECK_LAUNCH();
        }
    }
    dh_timing_end(h);
    return 0;
}

// Bytes that dh_project_f64_split needs to keep K (n x n) over the q + 2 passes of a
// solve, 0 where that does not pay.  A kept pass is bound by its workgroups' chunk
// by chunk reads where K is larger than the 256 MB cache and there is about one
// workgroup per CU; with two column blocks and up to 32 features a fused pass is as
// fast there, and forming K has to come back over the passes.  d = l = 16, fused ->
// kept: n = 8192 0.56 -> 0.63 ms (q = 0), 0.86 -> 0.90 (q = 1), 1.15 -> 1.14 (q = 2);
// n = 16384 1.94 -> 2.03 (q = 0), 2.98 -> 2.85 (q = 1).  On the other side: n = 5000 1.3x,
// 6000 and 10000 1.03x, 20000 1.2x, 65536 1.17x (q = 0); n = 8192 with l = 33 1.06x or d =
// 33 1.1x; up to 3.1x at d = 256; d > 256, where a pass forms K anyway, 1.1x to 3x.
size_t dh_kkeep_bytes(dh_handle_t h, int n, int d, int l, int q) {
    const size_t bytes = kept_bytes(n, n);
    if (d > 32 || l > 32 || bytes <= (256u << 20)) return bytes;
    const long tiles = dh_cdiv(n, 64);
    const int splits = dh_j_splits(h->num_cu, tiles, dh_cdiv(n, 32));
    const bool once = 4 * tiles * splits > 3L * h->num_cu && tiles * splits <= h->num_cu;
    return once && (q == 0 || (q == 1 && splits > 1)) ? 0 : bytes;
}

// Y (m x l) = K(Xi, Xj) O + beta Y with the fused kernel, the j range in
// `splits` parts (partials to P + z ystride, ld m, when splits > 1).
// With `pack`, Omega is first packed (labels folded in) into the kernel's LDS
// image in a workspace and staged by direct copies; without it (the
// allocation-free entry point) the kernel stages it through registers.  Both
// put the same values in LDS, so both give the same bits.
static int project_f64_fused(dh_handle_t h, int m, int n, int d, int l, const double* Xi,
                             int ldxi, const double* Xj, int ldxj, const double* ni,
                             const double* nj, const double* yi, const double* yj, double gamma,
                             const double* O, int ldo, double beta, double* Y, int ldy, int ncb,
                             int groups, int jps, int splits, long ystride, bool pack) {
    dim3 grid(dh_cdiv(m, 64), groups, splits);
    const d2v* Opk = nullptr;
    const int ncbp = groups * ncb;
    if (pack) DH_CHECK_STATUS(pack_omega_f64(h, n, l, ncbp, O, ldo, yj, &Opk));
#define DH_DK(K)                                                                              \
    dispatch_ncb<K>(h, ncb, grid, m, n, d, l, Xi, ldxi, Xj, ldxj, ni, nj, yi, yj, gamma, O, ldo, \
                    Opk, ncbp, beta, Y, ldy, jps, ystride)
    if (d <= 32) return DH_DK(8);
    if (d <= 64) return DH_DK(16);
    if (d <= 128) return DH_DK(32);
    return DH_DK(64);
#undef DH_DK
}

// Column blocking of the fused FP64 pass: ncb blocks per group.
static void f64_columns(int d, int l, int* ncb, int* groups) {
    const int ncb_total = dh_cdiv(l, 16);
    // Above 128 features the 17-block tile spills its accumulators: cap at 12.
    int g = dh_cdiv(ncb_total, d > 128 ? 12 : 17);
    *ncb = ncb_instance(dh_cdiv(ncb_total, g));
    *groups = dh_cdiv(ncb_total, *ncb);
}

// Whole j range in one launch; `pack` as in project_f64_fused (without it, no
// workspace for d <= 256).
int dh_project_f64_impl(dh_handle_t h, int m, int n, int d, int l, const double* Xi, int ldxi,
                        const double* Xj, int ldxj, const double* ni, const double* nj,
                        const double* yi, const double* yj, double gamma, const double* O,
                        int ldo, double beta, double* Y, int ldy, bool pack) {
    if (m == 0 || l == 0) return 0;
    if (n == 0)  // K has no columns: Y = beta Y
        return dh_gemm_impl<double>(h, false, false, m, l, 0, 1.0, O, 1, O, ldo, beta, Y, ldy, 0);
    if (d > 256)
        return project_f64_blocked(h, m, n, d, l, Xi, ldxi, Xj, ldxj, ni, nj, yi, yj, gamma, O,
                                   ldo, beta, Y, ldy, nullptr, 0);
    int ncb, groups;
    f64_columns(d, l, &ncb, &groups);
    return project_f64_fused(h, m, n, d, l, Xi, ldxi, Xj, ldxj, ni, nj, yi, yj, gamma, O, ldo,
                             beta, Y, ldy, ncb, groups, n, 1, 0, pack);
}

// K of one point set (d <= 256) in the kept layout.  Segments of up to 16 row
// tiles, fewer while that leaves less than four workgroups per CU.
static int form_sym_f64(dh_handle_t h, int n, int d, const double* X, int ldx, const double* nrm,
                        double gamma, void* keep) {
    const int nt = dh_cdiv(n, 64);
    int seg = 16;
    while (seg > 1 && (long)nt * nt / (2 * seg) < 4L * h->num_cu) seg /= 2;
    const dim3 grid(nt, dh_cdiv(nt, seg));
    dh_timing_begin(h);
#define DH_FORM(DK)                                                                           \
    form_sym_f64_kernel<DK><<<grid, 256, 0, h->stream>>>(n, d, X, ldx, nrm, gamma, seg,       \
                                                         (d2v*)keep, 4 * nt)
    if (d <= 32)
        DH_FORM(8);
    else if (d <= 64)
        DH_FORM(16);
    else if (d <= 128)
        DH_FORM(32);
    else
        DH_FORM(64);
#undef DH_FORM
    dh_timing_end(h);
    DH_CHECK_LAUNCH();
    return 0;
}

// Y = K O as dh_project_f64_impl with beta = 0; a grid of at most half a
// workgroup per CU splits the j range over more workgroups (partials in a
// workspace, summed in order).  The range finder's passes use it;
// dh_rbf_project_f64 keeps the one-launch form, so its allocation-free twin
// returns the same bits.  With `keep` (dh_kkeep_bytes; one point set, Xi = Xj)
// K is formed there first (kmode 1) or taken from there (kmode 2): same bits.
int dh_project_f64_split(dh_handle_t h, int m, int n, int d, int l, const double* Xi, int ldxi,
                         const double* Xj, int ldxj, const double* ni, const double* nj,
                         const double* yi, const double* yj, double gamma, const double* O,
                         int ldo, double* Y, int ldy, void* keep, int kmode) {
    if (m == 0 || l == 0) return 0;
    if (n == 0)
        return dh_project_f64_impl(h, m, n, d, l, Xi, ldxi, Xj, ldxj, ni, nj, yi, yj, gamma, O,
                                   ldo, 0.0, Y, ldy, true);
    if (d > 256)
        return project_f64_blocked(h, m, n, d, l, Xi, ldxi, Xj, ldxj, ni, nj, yi, yj, gamma, O,
                                   ldo, 0.0, Y, ldy, keep, kmode);
    int ncb, groups;
    f64_columns(d, l, &ncb, &groups);
    const int nch = dh_cdiv(n, 32);
    const int splits = dh_j_splits(h->num_cu, (long)dh_cdiv(m, 64) * groups, nch);
    const int jps = splits == 1 ? n : dh_cdiv(nch, splits) * 32;
    const long ystride = splits == 1 ? 0 : (long)m * l;
    double* P = Y;
    int ldp = ldy;
    if (splits > 1) {
        P = (double*)dh_ws(h, DH_WS_SPLITN, sizeof(double) * (size_t)ystride * splits);
        if (!P) return DH_ERR_ALLOC;
        ldp = m;
    }
    if (keep && kmode == 1) DH_CHECK_STATUS(form_sym_f64(h, n, d, Xi, ldxi, ni, gamma, keep));
    if (keep)
        DH_CHECK_STATUS(project_f64_kept(h, m, n, l, yi, yj, O, ldo, P, ldp, jps, splits, ystride,
                                         keep));
    else
        DH_CHECK_STATUS(project_f64_fused(h, m, n, d, l, Xi, ldxi, Xj, ldxj, ni, nj, yi, yj,
                                          gamma, O, ldo, 0.0, P, ldp, ncb, groups, jps, splits,
                                          ystride, true));
    if (splits == 1) return 0;
    sum_splits_f64_kernel<<<dh_cdiv(ystride, 256), 256, 0, h->stream>>>(m, l, splits, P, ystride,
                                                                        0.0, Y, ldy);
    DH_CHECK_LAUNCH();
    return 0;
}

extern "C" int dh_rbf_project_f64(dh_handle_t h, int m, int n, int d, int l, const double* Xi,
                                  int ldxi, const double* Xj, int ldxj, const double* yi,
                                  const double* yj, double gamma, const double* O, int ldo,
                                  double beta, double* Y, int ldy) {
    const char* name = "dh_rbf_project_f64";
    if (!h) return dh_fail(-1, "%s: NULL handle", name);
    if (m < 0) return dh_fail(-2, "%s: m < 0", name);
    if (n < 0) return dh_fail(-3, "%s: n < 0", name);
    if (d < 0) return dh_fail(-4, "%s: d < 0", name);
    if (l < 0) return dh_fail(-5, "%s: l < 0", name);
    if (ldxi < max(1, d)) return dh_fail(-7, "%s: ldxi < d", name);
    if (ldxj < max(1, d)) return dh_fail(-9, "%s: ldxj < d", name);
    if (ldo < max(1, n)) return dh_fail(-14, "%s: ldo < n", name);
    if (ldy < max(1, m)) return dh_fail(-17, "%s: ldy < m", name);
    if (m == 0 || l == 0) return 0;
    double* nrm = (double*)dh_ws(h, DH_WS_NORMS, sizeof(double) * ((size_t)m + n + 1));
    if (!nrm) return DH_ERR_ALLOC;
    DH_CHECK_STATUS(launch_sqnorms<double>(h, m, d, Xi, ldxi, nrm));
    DH_CHECK_STATUS(launch_sqnorms<double>(h, n, d, Xj, ldxj, nrm + m));
    return dh_project_f64_impl(h, m, n, d, l, Xi, ldxi, Xj, ldxj, nrm, nrm + m, yi, yj, gamma, O,
                               ldo, beta, Y, ldy, true);
}

// ------------------------------------------------------------ error pass
//
// Per 64 x 64 tile: S = Xi^T Xj (k over d) and P = Q_i W_j^T (k over l) in two
// MFMA accumulator sets, then sum (K - P)^2 and K^2 in FP64.  One pair of
// partial sums per workgroup, reduced in a fixed order by a second kernel.
__global__ __launch_bounds__(256) void lra_error_f64_kernel(
    int n, int d, int l, const double* __restrict__ X, int ldx, const double* __restrict__ nrm,
    const double* __restrict__ y, double gamma, const double* __restrict__ Q, int ldq,
    const double* __restrict__ W, int ldw, double* __restrict__ partial) {
    constexpr int BM = 64, BN = 64, FM = 2, FN = 2;
    __shared__ double sA[kTileBK][BM + kTilePad];
    __shared__ double sB[kTileBK][BN + kTilePad];
    __shared__ double red[2][4];
    const int m0 = blockIdx.x * BM, n0 = blockIdx.y * BN;
    dh_d4 S[FM][FN], P[FM][FN];
    zero_acc<double, FM, FN>(S);
    zero_acc<double, FM, FN>(P);
    tile_mma<double, BM, BN, true, false>(S, sA, sB, n, n, m0, n0, 0, d, X, ldx, X, ldx);
    tile_mma<double, BM, BN, false, true>(P, sA, sB, n, n, m0, n0, 0, l, Q, ldq, W, ldw);
    double se = 0.0, sk = 0.0;
#pragma unroll
    for (int a = 0; a < FM; ++a)
#pragma unroll
        for (int b = 0; b < FN; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                int i = m0 + tile_row<double, BM, BN>(a, r);
                int j = n0 + tile_col<BM, BN>(b);
                if (i < n && j < n) {
                    double d2 = nrm[i] + nrm[j] - 2.0 * S[a][b][r];
                    d2 = d2 > 0.0 ? d2 : 0.0;
                    double kv = exp(-gamma * d2);
                    if (y) kv *= y[i] * y[j];
                    double e = kv - P[a][b][r];
                    se += e * e;
                    sk += kv * kv;
                }
            }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        se += __shfl_xor(se, o);
        sk += __shfl_xor(sk, o);
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) {
        red[0][wave] = se;
        red[1][wave] = sk;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        size_t b = (size_t)blockIdx.y * gridDim.x + blockIdx.x;
        partial[2 * b] = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
        partial[2 * b + 1] = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
    }
}

// The same sums on 128 x 128 tiles of the upper triangle: distances and
// exponentials are symmetric, so tile (I, J) forms K once and compares it with
// Q_I W_J^T and, off the diagonal, with the transpose of Q_J W_I^T, in the
// same accumulator layout.  Operands are point-major copies padded to whole
// 16-deep stages of 128 bytes (pack_points_kernel, transpose_panel_kernel),
// staged by direct copies through a 3-deep LDS ring without a gap between the
// phases and tiles; 8 waves of 32 x 64, one persistent workgroup per CU.  A
// stage's 16-byte pieces of point i lie at p ^ ((i / 2) % 8) of its 128 bytes;
// lane group g takes pieces 2g and 2g + 1 as the k-slot g of four MFMAs.  Each
// lane adds its tiles' sums up with their rounding errors (two-sum), so how
// many tiles a lane gets does not matter to the result's accuracy.  At n =
// 65536, d = 128, l = 272: 50.2 ms, 57 TFLOP/s of the 2.9e12 that are left (73% of
// the FP64 MFMA peak; the 64 x 64 tiles 63%), the exponentials between them.
__global__ __launch_bounds__(512) void lra_error_sym_kernel(
    int n, int sd, int sl, const double* __restrict__ Xp, const double* __restrict__ nrm,
    const double* __restrict__ y, double gamma, int ntiles, double* __restrict__ partial) {
    __shared__ __align__(128) char ring[3][2][128 * 128];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, li = lane & 15;
    const int wi = wave & 3, wj = wave >> 2;
    const int dp = 16 * sd, lp = 16 * sl;
    const size_t qofs = (size_t)n * dp, wofs = (size_t)n * lp;  // Q after the points, W after Q
    // Tiles in order of columns bj, rows bi <= bj; each XCD a contiguous range.
    const int x = blockIdx.x & 7, per = ntiles / 8, rem = ntiles % 8;
    int tile = x * per + min(x, rem);
    const int last = tile + per + (x < rem ? 1 : 0), step = gridDim.x >> 3;
    tile += blockIdx.x >> 3;
    struct Tile {
        int i0, j0, nst;
    };
    auto decode = [&](int t) {
        int bj = (int)((sqrtf(8.0f * (float)t + 1.0f) - 1.0f) * 0.5f);
        while ((bj + 1) * (bj + 2) / 2 <= t) ++bj;
        while (bj * (bj + 1) / 2 > t) --bj;
        const int bi = t - bj * (bj + 1) / 2;
        return Tile{__builtin_amdgcn_readfirstlane(bi * 128),
                    __builtin_amdgcn_readfirstlane(bj * 128),
                    __builtin_amdgcn_readfirstlane(bi == bj ? sd + sl : sd + 2 * sl)};
    };
    const unsigned ring0 = (unsigned)(uintptr_t)(__attribute__((address_space(3))) char*)ring;
    int ftile = tile, fst = 0, fsl = 0;  // the next stage to copy, and its slot
    Tile f = decode(min(tile, ntiles - 1));
    unsigned ri[2], rj[2], off[2];  // this lane's rows from i0 / j0 and bytes within a stage
    auto rows = [&]() {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int row = 8 * (8 * u + wave) + (lane >> 3);
            ri[u] = (unsigned)(min(f.i0 + row, n - 1) - f.i0) * 8u;
            rj[u] = (unsigned)(min(f.j0 + row, n - 1) - f.j0) * 8u;
            off[u] = (unsigned)(((lane & 7) ^ ((row >> 1) & 7)) * 16);
        }
    };
    auto issue = [&]() {  // false once the last tile's stages are under way
        if (ftile >= last) return false;
        const bool dist = fst < sd, first = fst < sd + sl;
        // (Arithmetic instead of choices between captured values, which would be
        // kept in memory to be chosen by address.)
        const int pd = dist, pw = !dist && !first, pq = !dist && first;
        const int ld = lp + pd * (dp - lp);
        const int k0 = 16 * (fst - (1 - pd) * sd - pw * sl);
        const double* a = Xp + (size_t)(1 - pd) * qofs + (size_t)pw * wofs + (size_t)f.i0 * ld + k0;
        const double* b = Xp + (size_t)(1 - pd) * qofs + (size_t)pq * wofs + (size_t)f.j0 * ld + k0;
        const unsigned to = ring0 + 32768u * fsl + 1024u * wave;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            dma16_at(a, ri[u] * (unsigned)ld + off[u], to + 8192 * u);
            dma16_at(b, rj[u] * (unsigned)ld + off[u], to + 16384 + 8192 * u);
        }
        fsl = fsl == 2 ? 0 : fsl + 1;
        if (++fst == f.nst) {
            fst = 0;
            ftile += step;
            if (ftile < last) {
                f = decode(ftile);
                rows();
            }
        }
        return true;
    };
    const int off0 = ((2 * g) ^ (li >> 1)) * 16, off1 = ((2 * g + 1) ^ (li >> 1)) * 16;
    rows();
    issue();
    bool ahead = issue();  // a stage after the one to be waited for is under way
    int slot = 0;
    // acc = `count` stages of (J side) . (I side).
    auto product = [&](dh_d4(&acc)[4][2], int count) {
#pragma unroll
        for (int cj = 0; cj < 4; ++cj)
#pragma unroll
            for (int ci = 0; ci < 2; ++ci) acc[cj][ci] = dh_d4{0, 0, 0, 0};
        for (int st = 0; st < count; ++st) {
            if (ahead)
                __builtin_amdgcn_s_waitcnt(0x0F74);  // all but the newest stage's four copies
            else
                wait_vm();
            __syncthreads();
            ahead = issue();
            const char* la = ring[slot][0] + (wi * 32 + li) * 128;
            const char* lb = ring[slot][1] + (wj * 64 + li) * 128;
            slot = slot == 2 ? 0 : slot + 1;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int o = h ? off1 : off0;
                d2v av[2], bv[4];
#pragma unroll
                for (int c = 0; c < 2; ++c) av[c] = *(const d2v*)(la + c * 2048 + o);
#pragma unroll
                for (int c = 0; c < 4; ++c) bv[c] = *(const d2v*)(lb + c * 2048 + o);
#pragma unroll
                for (int e = 0; e < 2; ++e)
#pragma unroll
                    for (int cj = 0; cj < 4; ++cj)
#pragma unroll
                        for (int ci = 0; ci < 2; ++ci)
                            acc[cj][ci] = Mfma<double>::op(bv[cj][e], av[ci][e], acc[cj][ci]);
            }
        }
    };
    double se = 0.0, sk = 0.0, le = 0.0, lk = 0.0;  // sums and their rounding errors
    auto add = [](double& s, double& c, double v) {
        const double t = s + v, z = t - s;
        c += (s - (t - z)) + (v - z);
        s = t;
    };
    for (; tile < last; tile += step) {
        const Tile o = decode(tile);
        const int i1 = o.i0 + wi * 32 + li, j1 = o.j0 + wj * 64 + g;
        dh_d4 K[4][2], P[4][2];
        product(K, sd);
        double ni[2], yi[2], ts = 0.0;
#pragma unroll
        for (int ci = 0; ci < 2; ++ci) {
            const int i = min(i1 + 16 * ci, n - 1);
            ni[ci] = nrm[i];
            yi[ci] = y ? y[i] : 1.0;
        }
#pragma unroll
        for (int cj = 0; cj < 4; ++cj) {
            double nj[4], yj[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int j = min(j1 + 16 * cj + 4 * r, n - 1);
                nj[r] = nrm[j];
                yj[r] = y ? y[j] : 1.0;
            }
            wait_vm();  // here, so that no wait is left for the products' loop
#pragma unroll
            for (int ci = 0; ci < 2; ++ci)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    double d2 = ni[ci] + nj[r] - 2.0 * K[cj][ci][r];
                    d2 = d2 > 0.0 ? d2 : 0.0;
                    double kv = exp(-gamma * d2);
                    if (y) kv *= yi[ci] * yj[r];
                    K[cj][ci][r] = kv;
                    ts += (i1 + 16 * ci < n && j1 + 16 * cj + 4 * r < n) ? kv * kv : 0.0;
                }
        }
        const bool diag = o.i0 == o.j0;
        add(sk, lk, diag ? ts : 2.0 * ts);
        for (int side = 0; side < (diag ? 1 : 2); ++side) {
            product(P, sl);
            ts = 0.0;
#pragma unroll
            for (int cj = 0; cj < 4; ++cj)
#pragma unroll
                for (int ci = 0; ci < 2; ++ci)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const double e = K[cj][ci][r] - P[cj][ci][r];
                        ts += (i1 + 16 * ci < n && j1 + 16 * cj + 4 * r < n) ? e * e : 0.0;
                    }
            add(se, le, ts);
        }
    }
    // The error of an infinite sum is NaN: the sum stands without it.
    se += le == le ? le : 0.0;
    sk += lk == lk ? lk : 0.0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        se += __shfl_xor(se, o);
        sk += __shfl_xor(sk, o);
    }
    if (lane == 0) {
        double* p = partial + 2 * (8 * (size_t)blockIdx.x + wave);
        p[0] = se;
        p[1] = sk;
    }
}

// Points (d features each, ld ldx) as rows of dp features, zero-padded.
__global__ __launch_bounds__(256) void pack_points_kernel(int n, int d, int dp,
                                                          const double* __restrict__ X, int ldx,
                                                          double* __restrict__ out) {
    const size_t e = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= (size_t)n * dp) return;
    const int f = (int)(e % dp);
    out[e] = f < d ? X[f + (e / dp) * ldx] : 0.0;
}

// The n x l column-major panel P as rows of lp columns, zero-padded.
__global__ __launch_bounds__(256) void transpose_panel_kernel(int n, int l, int lp,
                                                              const double* __restrict__ P,
                                                              int ldp, double* __restrict__ out) {
    __shared__ double s[32][33];
    const int i0 = blockIdx.x * 32, c0 = blockIdx.y * 32, a = threadIdx.x & 31, b = threadIdx.x >> 5;
#pragma unroll
    for (int u = 0; u < 32; u += 8) {
        const int c = c0 + b + u, i = i0 + a;
        s[b + u][a] = (i < n && c < l) ? P[i + (size_t)c * ldp] : 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 32; u += 8) {
        const int i = i0 + b + u, c = c0 + a;
        if (i < n && c < lp) out[(size_t)i * lp + c] = s[a][b + u];
    }
}

// Fixed-order reduction of `count` (se, sk) pairs into out[0..1].
__global__ __launch_bounds__(256) void reduce_pairs_kernel(size_t count,
                                                            const double* __restrict__ partial,
                                                            double* __restrict__ out) {
    __shared__ double red[2][256];
    double se = 0.0, sk = 0.0;
    for (size_t b = threadIdx.x; b < count; b += 256) {
        se += partial[2 * b];
        sk += partial[2 * b + 1];
    }
    red[0][threadIdx.x] = se;
    red[1][threadIdx.x] = sk;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if (threadIdx.x < s) {
            red[0][threadIdx.x] += red[0][threadIdx.x + s];
            red[1][threadIdx.x] += red[1][threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[0] = red[0][0];
        out[1] = red[1][0];
    }
}

extern "C" int dh_lra_error(dh_handle_t h, int n, int d, int l, const double* X, int ldx,
                            const double* y, double gamma, const double* Q, int ldq,
                            const double* W, int ldw, double* err2) {
    const char* name = "dh_lra_error";
    if (!h) return dh_fail(-1, "%s: NULL handle", name);
    if (n < 0) return dh_fail(-2, "%s: n < 0", name);
    if (d < 0) return dh_fail(-3, "%s: d < 0", name);
    if (l < 0) return dh_fail(-4, "%s: l < 0", name);
    if (ldx < max(1, d)) return dh_fail(-6, "%s: ldx < d", name);
    if (ldq < max(1, n)) return dh_fail(-10, "%s: ldq < n", name);
    if (ldw < max(1, n)) return dh_fail(-12, "%s: ldw < n", name);
    if (!err2) return dh_fail(-13, "%s: err2 is NULL", name);
    err2[0] = err2[1] = 0.0;
    if (n == 0) return 0;
    double* nrm = (double*)dh_ws(h, DH_WS_NORMS, sizeof(double) * (size_t)n);
    if (!nrm) return DH_ERR_ALLOC;
    DH_CHECK_STATUS(launch_sqnorms<double>(h, n, d, X, ldx, nrm));
    // 128 x 128 tiles of one triangle from more than five per CU (n = 6401): there
    // the last, partly filled round of tiles no longer costs more than they
    // save (d = 20, l = 250: n = 5000 0.36 -> 0.37 ms, n = 8000 0.84 -> 0.71 ms; n = 65536,
    // d = 128, l = 272: 71.1 -> 50.0 ms).  The 64 x 64 tiles of the whole matrix below
    // that, for d = 0 or l = 0, and where the point-major copies cannot be had.  A
    // tile's copies have 32-bit byte offsets, a launch fewer than 2^32 threads.
    const int sd = dh_cdiv(d, 16), sl = dh_cdiv(l, 16), nt = dh_cdiv(n, 128);
    const long tiles = (long)nt * (nt + 1) / 2;
    double* Xp = nullptr;
    if (tiles > 5L * h->num_cu && d > 0 && l > 0 && std::max(sd, sl) < (1 << 18) &&
        tiles < (1L << 30) && (long)n * sd < (1L << 28) - 16)
        Xp = (double*)dh_ws(h, DH_WS_PACK64,
                            sizeof(double) * 16 * (size_t)n * ((size_t)sd + 2 * sl));
    const int wgs = (int)std::min<long>((tiles + 7) / 8 * 8, std::max(8, h->num_cu / 8 * 8));
    dim3 grid(dh_cdiv(n, 64), dh_cdiv(n, 64));
    size_t nblk = Xp ? 8 * (size_t)wgs : (size_t)grid.x * grid.y;
    double* part = (double*)dh_ws(h, DH_WS_PARTIAL, sizeof(double) * (2 * nblk + 2));
    if (!part) return DH_ERR_ALLOC;
    if (Xp) {
        double *Qp = Xp + 16 * (size_t)n * sd, *Wp = Qp + 16 * (size_t)n * sl;
        pack_points_kernel<<<(unsigned)(((size_t)n * sd * 16 + 255) / 256), 256, 0, h->stream>>>(
            n, d, 16 * sd, X, ldx, Xp);
        DH_CHECK_LAUNCH();
        const dim3 tg(dh_cdiv(n, 32), dh_cdiv(16 * sl, 32));
        transpose_panel_kernel<<<tg, 256, 0, h->stream>>>(n, l, 16 * sl, Q, ldq, Qp);
        DH_CHECK_LAUNCH();
        transpose_panel_kernel<<<tg, 256, 0, h->stream>>>(n, l, 16 * sl, W, ldw, Wp);
        DH_CHECK_LAUNCH();
        lra_error_sym_kernel<<<wgs, 512, 0, h->stream>>>(n, sd, sl, Xp, nrm, y, gamma,
                                                         (int)tiles, part);
    } else {
        lra_error_f64_kernel<<<grid, 256, 0, h->stream>>>(n, d, l, X, ldx, nrm, y, gamma, Q, ldq,
                                                          W, ldw, part);
    }
    DH_CHECK_LAUNCH();
    reduce_pairs_kernel<<<1, 256, 0, h->stream>>>(nblk, part, part + 2 * nblk);
    DH_CHECK_LAUNCH();
    DH_CHECK_HIP(hipMemcpyAsync(err2, part + 2 * nblk, 2 * sizeof(double), hipMemcpyDeviceToHost,
                                h->stream));
    DH_CHECK_HIP(hipStreamSynchronize(h->stream));
    return 0;
}
