// 16-bit range-finder passes on kept K values, for points of 129..256 features:
// one kernel forms K for all the passes of a solve, in the projection's operand
// layout, and a pass is then the projection alone.  The values are those of the fused kernels (the same
// products and epilogue), and so are the order of the chunks and the MFMAs: a
// solve returns the same bits either way.
//
// Layout: Kk[(t nrb + rb) 64 + L], the 16-byte A operand of lane L for 16-row
// block rb and 32-point chunk t; chunks outermost, because all waves walk them
// together.
#include "rbf16_kernels.h"

namespace {

template <int N>
__device__ __forceinline__ void wait_vm_but() {  // all but the newest N
    static_assert(N < 64, "vmcnt has six bits");
    __builtin_amdgcn_s_waitcnt(0x0F70 | (N & 15) | ((N >> 4) << 14));
}

// Forms K: 4 waves of 64 rows, the points of the column set through a 3-deep LDS
// ring of direct copies (as project_rows).  Grid: x = 256 rows, z = range of
// cps chunks.  Bound by the 2 bytes per entry it writes (n = 131072 with FP8
// distances: 9.1 ms, 3.8 TB/s).
template <int DK, bool F16, bool D8>
__global__ __launch_bounds__(256) void form16_kernel(
    int m, int nchunks, const bf16x8* __restrict__ Xi, const bf16x8* __restrict__ Xj,
    const float* __restrict__ ai, const float* __restrict__ bj, const float* __restrict__ si,
    const float* __restrict__ sj, float c2, int cps, int nrb, bf16x8* __restrict__ Kk) {
    using XS = XSlots<DK>;
    constexpr int XG = XS::XG, XROW = XS::XROW, WAVES = 4, RB = 4, NBUF = 3;
    __shared__ bf16x8 sX[NBUF][XS::SLOTS];
    __shared__ float sB[NBUF][64], sS[D8 ? NBUF : 1][64];
    const int t0 = blockIdx.z * cps, last = min(cps, nchunks - t0) - 1;
    Xj += (size_t)t0 * 32 * XG;
    bj += (size_t)t0 * 32;
    if (D8) sj += (size_t)t0 * 32;
    const int lane = threadIdx.x & 63, g = lane >> 4, li = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int rb0 = (blockIdx.x * WAVES + wave) * RB;
    auto grp = [&](int q) { return D8 ? 8 * (q >> 1) + 2 * g + (q & 1) : 4 * q + g; };
    bf16x8 xb[RB][DK];
    float arow[RB], crow[RB];
    f32x4 ainit[RB];
#pragma unroll
    for (int ib = 0; ib < RB; ++ib) {
        const int row = (rb0 + ib) * 16 + li;
#pragma unroll
        for (int q = 0; q < DK; ++q) {
            bf16x8 z = {};
            xb[ib][q] = (row < m) ? Xi[(size_t)row * XG + grp(q)] : z;
        }
        arow[ib] = (row < m) ? ai[row] : 0.f;
        crow[ib] = D8 ? c2 * ((row < m) ? si[row] : 0.f) : c2;
        const float v = (D8 || c2 == 0.f) ? 0.f : arow[ib] / c2;
        ainit[ib] = f32x4{v, v, v, v};
    }
    constexpr int NXK = (XS::INSTR + WAVES - 1) / WAVES;
    unsigned offx[NXK];
#pragma unroll
    for (int k = 0; k < XS::INSTR; k += WAVES) {
        int slot = (k + wave) * 64 + lane, row = slot / XROW, col = slot % XROW;
        if (row >= 32 || col >= XG) {
            row = 0;
            col = 0;
        }
        offx[k / WAVES] = (unsigned)(row * XG + col) * 16u;
    }
    auto stage = [&](int t, int buf) {
        const bf16x8* xc = Xj + (size_t)t * 32 * XG;
#pragma unroll
        for (int k = 0; k < XS::INSTR; k += WAVES) {
            const int kk = k + wave;
            if (XS::INSTR % WAVES == 0 || kk < XS::INSTR)
                dma16(xc, offx[k / WAVES], &sX[buf][kk * 64]);
        }
        if (wave == WAVES - 1) dma4(bj + (size_t)t * 32, (unsigned)(lane & 31) * 4u, &sB[buf][0]);
        if (D8 && wave == WAVES - 2)
            dma4(sj + (size_t)t * 32, (unsigned)(lane & 31) * 4u, &sS[D8 ? buf : 0][0]);
    };
    bf16x8* kp = Kk + ((size_t)t0 * nrb + rb0) * 64 + lane;
    stage(0, 0);
    wait_vm();
    int buf = 0;
    for (int t = 0; t <= last; ++t) {
        const int nbuf = buf == NBUF - 1 ? 0 : buf + 1;
        wait_vm_but<RB>();  // the copies of chunk t; the stores after them may be under way
        __syncthreads();
        stage(min(t + 1, last), nbuf);
        f32x4 s[2][RB];
        bf16x8 kb[RB];
#pragma unroll
        for (int jb = 0; jb < 2; ++jb) {
            bf16x8 a[DK];
#pragma unroll
            for (int q = 0; q < DK; ++q) a[q] = sX[buf][(16 * jb + li) * XROW + grp(q)];
#pragma unroll
            for (int ib = 0; ib < RB; ++ib) s[jb][ib] = ainit[ib];
            if constexpr (D8) {
#pragma unroll
                for (int q = 0; q < DK; q += 2)
#pragma unroll
                    for (int ib = 0; ib < RB; ++ib)
                        s[jb][ib] = mfma_fp8(join16(a[q], a[q + 1]),
                                             join16(xb[ib][q], xb[ib][q + 1]), s[jb][ib]);
            } else {
#pragma unroll
                for (int q = 0; q < DK; ++q)
#pragma unroll
                    for (int ib = 0; ib < RB; ++ib)
                        s[jb][ib] = mfma16<F16>(a[q], xb[ib][q], s[jb][ib]);
            }
        }
        // The values of project_rows' epilogue: element 4 jb + r.
#pragma unroll
        for (int jb = 0; jb < 2; ++jb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float bv = sB[buf][16 * jb + 4 * g + r];
                const float sj = D8 ? sS[D8 ? buf : 0][16 * jb + 4 * g + r] : 1.f;
#pragma unroll
                for (int ib = 0; ib < RB; ++ib) {
                    const float cc = D8 ? crow[ib] * sj : crow[ib];
                    const float e = __builtin_amdgcn_exp2f(
                        fmaf(cc, s[jb][ib][r], D8 ? arow[ib] + bv : bv));
                    kb[ib][4 * jb + r] = to16<F16>(__builtin_amdgcn_fmed3f(e, 0.f, 1.f));
                }
            }
#pragma unroll
        for (int ib = 0; ib < RB; ++ib) kp[ib * 64] = kb[ib];
        kp += (size_t)nrb * 64;
        buf = nbuf;
    }
    wait_vm();
}

// One pass: Y = K Op.  A workgroup of 8 waves takes RS row slots of 64 rows and
// NO column blocks (one group, or two adjacent ones where the rows of K are then
// read once for both); the 8 / RS waves of a row slot share out the columns, CB or
// CB - 1 blocks each.  64 rows to a wave halve its reads of Omega from LDS, whose
// bandwidth bounds the pass with 32 rows and all 17 blocks per wave; 64 rows and
// 17 blocks would be 272 accumulators.  Waves w and w + 4 share a SIMD, so the
// larger shares go to waves 0..3.  K and Omega go through an LDS ring of direct
// copies, NBUF - 1 chunks ahead; one barrier per chunk.  At n = 65536, l = 272:
// 2.27 ms (2.41 ms with 32 rows and all blocks per wave), between the 1.6 ms of
// reading K and the clock that power leaves beside it.
template <int NO, int RS, bool F16>
__global__ __launch_bounds__(512, 1) void kept_project16_kernel(
    int m, int nchunks, int l, int ncb_total, const bf16x8* __restrict__ Kk, int nrb,
    const bf16x8* __restrict__ Op, const double* __restrict__ yi, double* __restrict__ Y, int ldy,
    int cps, long ystride) {
    constexpr int WAVES = 8, RB = 4, CS = WAVES / RS, CB = (NO + CS - 1) / CS;
    constexpr int NBUF = NO > 17 ? 3 : 4, KW = RS * RB / WAVES;
    constexpr int BIG = NO - CS * (CB - 1);  // column shares of CB blocks
    static_assert(RS * RB % WAVES == 0, "K copies split evenly");
    static_assert(BIG * RS >= 4 || BIG == CS, "larger shares on waves 0..3");
    __shared__ bf16x8 sO[NBUF][NO * 64];
    __shared__ bf16x8 sK[NBUF][RS * RB * 64];
    const int lane = threadIdx.x & 63, g = lane >> 4, li = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int wrow = wave % RS, share = wave / RS;
    const bool big = share < BIG;
    const int wcb = share * CB - max(0, share - BIG);  // first block of the share
    const int cb0 = blockIdx.y * NO + wcb;
    const int t0 = blockIdx.z * cps, last = min(cps, nchunks - t0) - 1;
    const bf16x8* kbase = Kk + ((size_t)t0 * nrb + blockIdx.x * RS * RB) * 64;
    const bf16x8* obase = Op + ((size_t)t0 * ncb_total + blockIdx.y * NO) * 64;
    Y += blockIdx.z * ystride;
    auto stage = [&](int t, int buf) {
        const bf16x8* kc = kbase + (size_t)t * nrb * 64;
        const bf16x8* oc = obase + (size_t)t * ncb_total * 64;
#pragma unroll
        for (int k = 0; k < KW; ++k)
            dma16(kc + (k * WAVES + wave) * 64, (unsigned)lane * 16u,
                  &sK[buf][(k * WAVES + wave) * 64]);
#pragma unroll
        for (int k = 0; k < NO; k += WAVES) {
            const int kk = k + wave;
            if (NO % WAVES == 0 || kk < NO)
                dma16(oc + kk * 64, (unsigned)lane * 16u, &sO[buf][kk * 64]);
        }
    };
    f32x4 acc[RB][CB];
#pragma unroll
    for (int ib = 0; ib < RB; ++ib)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) acc[ib][cb] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int b = 0; b < NBUF - 1; ++b) stage(min(b, last), b);
    int buf = 0;
    for (int t = 0; t <= last; ++t) {
        // Waves below NO % WAVES copy one block more per chunk.
        if (wave < NO % WAVES)
            wait_vm_but<(NBUF - 2) * (KW + NO / WAVES + 1)>();
        else
            wait_vm_but<(NBUF - 2) * (KW + NO / WAVES)>();
        __syncthreads();
        stage(min(t + NBUF - 1, last), buf == 0 ? NBUF - 1 : buf - 1);
        bf16x8 kb[RB], bo[CB];
#pragma unroll
        for (int ib = 0; ib < RB; ++ib) kb[ib] = sK[buf][(wrow * RB + ib) * 64 + lane];
        const bf16x8* so = &sO[buf][wcb * 64 + lane];
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
            if (cb < CB - 1 || big) bo[cb] = so[cb * 64];
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
            if (cb < CB - 1 || big)
#pragma unroll
                for (int ib = 0; ib < RB; ++ib)
                    acc[ib][cb] = mfma16<F16>(kb[ib], bo[cb], acc[ib][cb]);
        buf = buf == NBUF - 1 ? 0 : buf + 1;
    }
    wait_vm();  // the copies ahead of the end still write this workgroup's LDS
#pragma unroll
    for (int ib = 0; ib < RB; ++ib)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int i = ((blockIdx.x * RS + wrow) * RB + ib) * 16 + 4 * g + r;
                const int c = 16 * (cb0 + cb) + li;
                if (i < m && c < l && (cb < CB - 1 || big)) {
                    double v = (double)acc[ib][cb][r];
                    if (yi) v *= yi[i];
                    Y[i + (size_t)c * ldy] = v;
                }
            }
}

}  // namespace

// Row blocks of the layout: whole workgroups of 256 rows.
static int kept_row_blocks(int m) { return dh_cdiv(m, 256) * 16; }

size_t dh_kept16_bytes(int m, int nchunks) {
    return sizeof(bf16x8) * 64 * (size_t)kept_row_blocks(m) * (size_t)nchunks;
}

// A kept pass costs about the same at every feature count (its reading of K), so
// keeping K pays where the fused pass is slow: at 256 features, whose Xi
// fragments leave 16-bit distances 32 rows for each of four waves, and whose FP8
// distances pair up or carry few columns, and over at least three passes, for
// the forming of K.  Solves with q = 1, fused -> kept: FP16 n = 65536, l = 138: 10.1
// -> 7.8 ms, l = 272: 15.6 -> 10.8 ms, l = 544: 33.3 -> 22.1 ms; FP8 n = 16384, l = 138: 2.11
// -> 1.56 ms, l = 544: 4.76 -> 4.46 ms, n = 65536, l = 544: 21.9 -> 21.0 ms (n = 131072 73.1
// -> 72.1, within the runs' range; q = 2 98.9 -> 94.8).  16-bit distances at few points
// do not pay for the forming and its launch: l = 138 from n = 8192 on (1.04x; n = 2048 to
// 4096 0.98x, 6000 1.00x), 17 column blocks above it (l = 272, n = 8500 to 11500 1.02x to
// 1.05x; n = 2048 to 6000 0.96x to 0.98x, 8192 0.99x).  Also not: FP8 at l = 272 9.7 ->
// 10.0 ms, two passes of BF16 2.8 -> 2.7 ms, FP16 at 128 features 9.8 -> 10.1 ms (q = 2:
// 13.2 -> 13.0 ms).
bool dh_kept16_pays(int n, int dpad, bool fp8, int ncb, int groups, int passes) {
    if (dpad != 256 || passes < 3) return false;
    if (fp8) return ncb == 9 || (ncb == 17 && groups % 2 == 0);
    return (ncb == 9 && n >= 8192) || (ncb == 17 && n > 8192);
}

// Whether one solve alone gains more than allocating and freeing a buffer takes
// (about 0.3 ms above 64 MB): with a handle per solve and a new buffer each, FP16 l =
// 138, q = 1 n = 8200 1.69 ms and 1.48 without, n = 12000 1.60 and 1.69.
bool dh_kept16_fresh(int n, size_t bytes) { return bytes <= (64u << 20) || n >= 12000; }

int dh_form16(dh_handle_t h, bool f16, bool fp8, int dpad, int m, int nchunks, const bf16x8* Xi,
              const bf16x8* Xj, const float* ai, const float* bj, const float* si,
              const float* sj, float c2, void* keep) {
    const int nrb = kept_row_blocks(m), gx = nrb / 16;
    const int cps = dh_cdiv(nchunks, std::max(1, std::min(nchunks, 4 * h->num_cu / gx)));
    const dim3 grid(gx, 1, dh_cdiv(nchunks, cps));
#define DH_FORM(DK, F16, D8)                                                                \
    form16_kernel<DK, F16, D8><<<grid, 256, 0, h->stream>>>(m, nchunks, Xi, Xj, ai, bj, si, \
                                                            sj, c2, cps, nrb, (bf16x8*)keep)
    if (dpad != 256)
        return dh_fail(DH_ERR_UNSUPPORTED, "kept K: no kernel for %d features", dpad);
    dh_timing_begin(h);
    if (fp8)
        DH_FORM(4, false, true);
    else if (f16)
        DH_FORM(8, true, false);
    else
        DH_FORM(8, false, false);
    dh_timing_end(h);
#undef DH_FORM
    DH_CHECK_LAUNCH();
    return 0;
}

int dh_project16_kept(dh_handle_t h, bool f16, int ncb, int groups, int m, int nchunks, int l,
                      int ncb_total, const void* keep, const bf16x8* Op, const double* yi,
                      double* Y, int ldy, int splits, long ystride) {
    const int nrb = kept_row_blocks(m), cps = dh_cdiv(nchunks, splits);
    const int nz = dh_cdiv(nchunks, cps);
    const bool pair = ncb == 17 && groups % 2 == 0;
    const dim3 grid(nrb / 16 * (pair ? 2 : 1), pair ? groups / 2 : groups, nz);
#define DH_KEPT(NO, RS)                                                                     \
    if (f16)                                                                                \
        kept_project16_kernel<NO, RS, true><<<grid, 512, 0, h->stream>>>(                   \
            m, nchunks, l, ncb_total, (const bf16x8*)keep, nrb, Op, yi, Y, ldy, cps, ystride); \
    else                                                                                    \
        kept_project16_kernel<NO, RS, false><<<grid, 512, 0, h->stream>>>(                  \
            m, nchunks, l, ncb_total, (const bf16x8*)keep, nrb, Op, yi, Y, ldy, cps, ystride)
    if (pair) {
        DH_KEPT(34, 2);
    } else if (ncb == 17) {
        DH_KEPT(17, 4);
    } else if (ncb == 9) {
        DH_KEPT(9, 4);
    } else {
        return dh_fail(DH_ERR_UNSUPPORTED, "kept K: no kernel for %d column blocks", ncb);
    }
#undef DH_KEPT
    DH_CHECK_LAUNCH();
    return 0;
}
