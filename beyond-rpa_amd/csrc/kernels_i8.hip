// Split-int8 Pi(u) build on gfx950 int8 MFMA (v_mfma_i32_16x16x64_i8).
//
// X_w = diag(sqrt(c_w)) R.  Column P of X_w gets one scale over all K rows,
// s_P = max_k |X_w[k][P]| / 127, and every element is written as
//   X = s_P (n0 + n1 2^-7 + n2 2^-14 + n3 2^-21),
// |n0| <= 127, |n1|, |n2|, |n3| <= 64 (each remainder is at most 1/2 before
// the 2^7 step), all four stored as int8.  The truncation is below 2^-28
// relative to the column maximum.  Pi_w[p][q] = s_p s_q sum_k x_p x_q and the
// ten slice products of level a + b <= 3 go to four int32 accumulators
//   L0 = n0 n0,  L1 = n0 n1 + n1 n0,  L2 = n0 n2 + n1 n1 + n2 n0,
//   L3 = n0 n3 + n1 n2 + n2 n1 + n3 n0,
// which are exact over the whole K: |L3| <= K (2*127*64 + 2*64*64) < 2^31 for
// K <= 87000 (the library caps K at 65536).  One FP64 combination per element,
//   Pi = s_p s_q (L0 + L1 2^-7 + L2 2^-14 + L3 2^-21),
// ends the product; the dropped level >= 4 products are ~2^-28 relative.
// The diagonal (and so tr Pi) is replaced by its exact double-double value
// from the column pass.
//
//   k_colscale_i8  s_w[P] and the exact diagonal, one pass over R for all w
//   k_split_i8     int8 slices of X_w, one read of R for all w
//   k_syrk_i8_128  128x128 output tiles, 8 waves of 64x32, int8 MFMA
//   k_syrk_i8_64   64x64 output tiles, 2 waves
#include "device_common.h"
#include "internal.h"

#define LAUNCH_CHECK(ctx)                                                                      \
    do {                                                                                       \
        hipError_t _e = hipGetLastError();                                                     \
        if (_e != hipSuccess)                                                                  \
            return brpa_fail((ctx), BRPA_ERR_HIP, "kernel launch failed: %s (%s:%d)",          \
                             hipGetErrorString(_e), __FILE__, __LINE__);                       \
    } while (0)

typedef __attribute__((address_space(1))) const double gdbl_t;
typedef int v4i_t __attribute__((ext_vector_type(4)));

// ---------------------------------------------------------------------------
// Column pass.  For each (w, P): scale8 = max_k |sqrt(c_w(k)) R[k][P]| / 127 and
// diag = sum_k c_w(k) R[k][P]^2 in double-double (rpa_CC.f90:444-447 sums the
// trace in REAL(F128)).  Work-groups per fragment: ceil(K/512) row chunks x
// ceil(N/64) column groups; a lane holds one column, each wave walks a quarter
// of the chunk's rows eight at a time, and the two tables come as scalar loads
// (the row is the same for the whole wave).  Frequencies in groups of 8: their
// maxima and sums stay in 48 registers.  The four waves are combined in LDS in
// wave order, and k_colscale_fin_i8 adds the chunks in order.
//
// Bound by FP64 VALU work (about 13 operations per element and frequency).
// At K = 10800, N = 1800, 24 frequencies the two kernels take 350 us; one
// work-group per 64 columns over all of K kept 29 of 256 CUs busy there (4809 us).
// Over 32 fragments of the batch shapes: 1361 us, before 3359.
constexpr int CS_WG = 16;       // frequencies per group of the split pass
constexpr int KS8 = 64;         // k-values (bytes) per stage and slice of the product
constexpr int CSF = 8;          // frequencies per register group of the column pass
constexpr int CSR = 8;          // rows per step of a wave
typedef __attribute__((address_space(4))) const double cdbl_t;

__global__ __launch_bounds__(256) void k_colscale_i8(const FragDev *__restrict__ fr,
                                                    const int64_t *__restrict__ pre, int nfrag) {
    __shared__ int64_t s_pre[FIND_LDS_MAX + 1];
    __shared__ double sM[4][4][64], sH[4][4][64], sL[4][4][64];
    const int64_t b = blockIdx.x;
    const int f = __builtin_amdgcn_readfirstlane(find_frag_lds(pre, nfrag, b, s_pre));
    const FragDev &F = fr[f];
    const int N = F.N, K = F.K, nF = F.F;
    const int ncg = (N + 63) / 64;
    const int lb = __builtin_amdgcn_readfirstlane(
        (int)(b - (nfrag <= FIND_LDS_MAX ? s_pre[f] : pre[f])));
    const int ck = lb / ncg, P0 = (lb - ck * ncg) * 64;
    const int c = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int P = P0 + c;
    const bool colok = P < N;
    const gdbl_t *R = (const gdbl_t *)F.R + (colok ? P : 0);
    const int kb = ck * CS_ROWS + wave * (CS_ROWS / 4), ke = min(K, kb + CS_ROWS / 4);
    for (int w0 = 0; w0 < nF; w0 += CSF) {
        const int nw = min(CSF, nF - w0);
        const cdbl_t *SD = (const cdbl_t *)(uintptr_t)F.sdtab + (int64_t)w0 * K;
        const cdbl_t *CD = (const cdbl_t *)(uintptr_t)F.dtab + (int64_t)w0 * K;
        double m[CSF], hi[CSF], lo[CSF];
#pragma unroll
        for (int i = 0; i < CSF; ++i) m[i] = hi[i] = lo[i] = 0.0;
        auto step = [&](double x, double r2, double r2e, double sd, double cw, int i) {
            m[i] = fmax(m[i], fabs(x * sd));
            const double p = cw * r2, pe = fma(cw, r2, -p) + cw * r2e;
            // TwoSum of hi and p; the errors collect in lo
            const double s = hi[i] + p, bb = s - hi[i];
            lo[i] += ((hi[i] - (s - bb)) + (p - bb)) + pe;
            hi[i] = s;
        };
        int k = kb;
        for (; k + CSR <= ke; k += CSR) {
            double x[CSR], r2[CSR], r2e[CSR];
#pragma unroll
            for (int r = 0; r < CSR; ++r) x[r] = R[(int64_t)(k + r) * N];
#pragma unroll
            for (int r = 0; r < CSR; ++r) {
                r2[r] = x[r] * x[r];
                r2e[r] = fma(x[r], x[r], -r2[r]);
            }
#pragma unroll
            for (int i = 0; i < CSF; ++i)
                if (i < nw) {
#pragma unroll
                    for (int r = 0; r < CSR; ++r)
                        step(x[r], r2[r], r2e[r], SD[i * K + k + r], CD[i * K + k + r], i);
                }
        }
        for (; k < ke; ++k) {
            const double x = R[(int64_t)k * N], r2 = x * x, r2e = fma(x, x, -r2);
#pragma unroll
            for (int i = 0; i < CSF; ++i)
                if (i < nw) step(x, r2, r2e, SD[i * K + k], CD[i * K + k], i);
        }
        // combine the four waves, four frequencies at a time
#pragma unroll
        for (int i0 = 0; i0 < CSF; i0 += 4) {
            __syncthreads();
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                sM[wave][i][c] = m[i0 + i];
                sH[wave][i][c] = hi[i0 + i];
                sL[wave][i][c] = lo[i0 + i];
            }
            __syncthreads();
            const int w = w0 + i0 + wave;
            if (w < nF && colok) {
                const double mm = fmax(fmax(sM[0][wave][c], sM[1][wave][c]),
                                       fmax(sM[2][wave][c], sM[3][wave][c]));
                dd_t t = {sH[0][wave][c], sL[0][wave][c]};
#pragma unroll
                for (int q = 1; q < 4; ++q) t = dd_add(t, (dd_t){sH[q][wave][c], sL[q][wave][c]});
                double *o = F.dpart + (((int64_t)ck * nF + w) * N + P) * 3;
                o[0] = mm;
                o[1] = t.hi;
                o[2] = t.lo;
            }
        }
    }
}

// scale8 and diag from the row chunks' partials, in chunk order.  Work-groups
// per fragment: ceil(F*N/256).
__global__ __launch_bounds__(256) void k_colscale_fin_i8(const FragDev *__restrict__ fr,
                                                        const int64_t *__restrict__ pre,
                                                        int nfrag) {
    const int64_t b = blockIdx.x;
    const int f = find_frag(pre, nfrag, b);
    const FragDev &F = fr[f];
    const int64_t e = (b - pre[f]) * 256 + threadIdx.x, FN = (int64_t)F.F * F.N;
    if (e >= FN) return;
    const int nck = (F.K + CS_ROWS - 1) / CS_ROWS;
    double m = 0.0;
    dd_t t = {0.0, 0.0};
    for (int q = 0; q < nck; ++q) {
        const double *o = F.dpart + ((int64_t)q * FN + e) * 3;
        m = fmax(m, o[0]);
        t = dd_add(t, (dd_t){o[1], o[2]});
    }
    F.scale8[e] = m / 127.0;
    F.diag[e] = t.hi + t.lo;
}

int launch_colscale_i8(brpa_ctx *ctx, const FragDev *fr, const int64_t *pre, int nfrag,
                       int64_t total, const int64_t *pre_fin, int64_t total_fin) {
    if (total <= 0) return BRPA_OK;
    hipLaunchKernelGGL(k_colscale_i8, dim3((unsigned)total), dim3(256), 0, ctx->stream, fr, pre,
                       nfrag);
    LAUNCH_CHECK(ctx);
    hipLaunchKernelGGL(k_colscale_fin_i8, dim3((unsigned)total_fin), dim3(256), 0, ctx->stream, fr,
                       pre_fin, nfrag);
    LAUNCH_CHECK(ctx);
    return BRPA_OK;
}

// ---------------------------------------------------------------------------
// Split pass.  Work-groups per fragment: (Kpad8 / 128) * ceil(N/64).  A
// 128-row x 64-column tile of R is staged in LDS once and sliced for every
// frequency.  Thread -> column tid/4, rows 32 (tid%4) .. +32, so each
// (w, slice, column) row segment of 128 bytes is written by 4 neighbouring
// threads.  Rows k >= K and columns past N write zeros / nothing.
// Bound by the writes of the slices: at K = 10800, N = 1800, 24 frequencies 440 us, 4.2
// TB/s (489 us with a rounding, a conversion and a scaling per slice and the four row
// quarters' tables on the same banks); 32 fragments of the batch shapes 2.94 ms (3.20).
__global__ __launch_bounds__(256) void k_split_i8(const FragDev *__restrict__ fr,
                                                 const int64_t *__restrict__ pre, int nfrag) {
    __shared__ int64_t s_pre[FIND_LDS_MAX + 1];
    // sqrt(c_w) of this work-group's rows; the four row quarters that a wave reads at once are
    // padded onto different banks
    constexpr int SQ = I8_KB / 4 + 2;
    __shared__ __attribute__((aligned(16))) double sSD[CS_WG][4 * SQ];
    const int64_t b = blockIdx.x;
    const int f = find_frag_lds(pre, nfrag, b, s_pre);
    const FragDev &F = fr[f];
    const int N = F.N, K = F.K;
    const int ncc = (N + 63) / 64;
    const int64_t lb = b - (nfrag <= FIND_LDS_MAX ? s_pre[f] : pre[f]);
    const int kc = (int)(lb / ncc), cc = (int)(lb - (int64_t)kc * ncc);
    const int k0 = kc * I8_KB, P0 = cc * 64;
    const int tid = threadIdx.x;
    const gdbl_t *R = (const gdbl_t *)F.R;
    const gdbl_t *SD = (const gdbl_t *)F.sdtab;
    // thread -> column P0 + tid/4 and its 32 rows 32 (tid%4) .. +32, held in registers
    const int c = tid >> 2, r0 = (tid & 3) * 32;
    const int P = P0 + c;
    const bool colok = P < N;
    double x[32];
#pragma unroll
    for (int j = 0; j < 32; ++j) {
        const int k = k0 + r0 + j;
        const bool ok = colok && k < K;
        x[j] = R[ok ? (int64_t)k * N + P : 0];
        x[j] = ok ? x[j] : 0.0;
    }
    const int64_t Kp = F.Kpad8;
    for (int w0 = 0; w0 < F.F; w0 += CS_WG) {
        const int nw = min(CS_WG, F.F - w0);
        __syncthreads();
        for (int e = tid; e < CS_WG * I8_KB; e += 256) {
            const int i = e / I8_KB, r = e - i * I8_KB;
            const bool ok = i < nw && k0 + r < K;
            const double v = SD[ok ? (int64_t)(w0 + i) * K + k0 + r : 0];
            sSD[i][r / 32 * SQ + r % 32] = ok ? v : 0.0;
        }
        __syncthreads();
        if (!colok) continue;
        for (int i = 0; i < nw; ++i) {
            const int w = w0 + i;
            const double sc = F.scale8[(int64_t)w * N + P];
            const double inv = sc > 0.0 ? 1.0 / sc : 0.0;
            uint32_t pk[NSLICE][8];
#pragma unroll
            for (int q = 0; q < 8; ++q) {
                uint32_t byte[NSLICE][4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int j = 4 * q + u;
                    double t = x[j] * sSD[i][(tid & 3) * SQ + j] * inv;   // |t| <= 127 (up to rounding)
                    // rounded to a multiple of 128^-s by adding 1.5 2^(52-7s), which leaves that
                    // multiple in the sum's low bits; every step is exact
#pragma unroll
                    for (int s = 0; s < NSLICE; ++s) {
                        const double M = 1.5 * (double)(1ull << (52 - 7 * s)), r = t + M;
                        t -= r - M;
                        byte[s][u] = (uint32_t)__double_as_longlong(r);
                    }
                }
#pragma unroll
                for (int s = 0; s < NSLICE; ++s) {
                    // the low bytes of four words
                    const uint32_t lo = __builtin_amdgcn_perm(byte[s][1], byte[s][0], 0x0c0c0400u),
                                   hi = __builtin_amdgcn_perm(byte[s][3], byte[s][2], 0x04000c0cu);
                    pk[s][q] = lo | hi;
                }
            }
#pragma unroll
            for (int s = 0; s < NSLICE; ++s) {
                int8_t *dst = F.sl8 + ((int64_t)w * NSLICE + s) * N * Kp +
                              ((int64_t)((k0 + r0) / KS8) * N + P) * KS8 + r0 % KS8;
                uint4 *d4 = reinterpret_cast<uint4 *>(dst);
                d4[0] = make_uint4(pk[s][0], pk[s][1], pk[s][2], pk[s][3]);
                d4[1] = make_uint4(pk[s][4], pk[s][5], pk[s][6], pk[s][7]);
            }
        }
    }
}

int launch_split_i8(brpa_ctx *ctx, const FragDev *fr, const int64_t *pre, int nfrag,
                    int64_t total) {
    if (total <= 0) return BRPA_OK;
    hipLaunchKernelGGL(k_split_i8, dim3((unsigned)total), dim3(256), 0, ctx->stream, fr, pre,
                       nfrag);
    LAUNCH_CHECK(ctx);
    return BRPA_OK;
}

// ---------------------------------------------------------------------------
// Product.  One TxT output tile pair (p-tile >= q-tile) of one frequency per
// work-group; work-groups per fragment: F * npairs(ceil(N/T)).  The waves
// own 64x32 sub-tiles: T = 128 -> 8 waves (2 x 4), T = 64 -> 2 waves (1 x 2).
// Only the lower triangle of Pi is written (the Cholesky reads no other).
//
// The slices lie in memory as [w][slice][k / 64][column][64], so that the 16 columns
// of a wave load are one contiguous KB (with the whole K of a column contiguous they
// were 16 half cache lines: 6-9 % slower).
//
// v_mfma_i32_16x16x64_i8 lane layout (lane l, 16 bytes per operand):
//   A[m = l%16][k = 16*(l/16) .. +15], B[k = 16*(l/16) .. +15][n = l%16],
//   D: 4 ints, D[r] = C[m = 4*(l/16) + r][n = l%16].
// Both operands are columns of X (k contiguous per column, 64 bytes = one
// MFMA k-depth per stage and slice), read from LDS the same way.
//
// Stages go straight from HBM to LDS (global_load_lds_dwordx4, 16 bytes per
// lane), double-buffered.  One wave load fills 1 KB = 16 columns x 64 bytes;
// lane l lands in column l/4, slot l%4, and fetches k-piece
// (l%4) ^ ((l/16)%4) of that column, so that the MFMA operand reads (16
// columns at one k-piece per 16 lanes) hit 16 distinct 4-bank groups.

typedef __attribute__((address_space(3))) void lds_void_t;

__device__ __forceinline__ int swz8(int col_local, int piece) {
    return piece ^ ((col_local >> 2) & 3);
}

__global__ __launch_bounds__(128) void k_syrk_i8_64(
    const FragDev *__restrict__ fr, const int64_t *__restrict__ pre, int nfrag) {
    constexpr int T = 64;
    constexpr int WJN = T / 32;                 // waves along columns
    constexpr int NW = (T / 64) * WJN;          // waves
    constexpr int GPS = T / 16;                 // 16-column groups per side and slice
    constexpr int LPS = NSLICE * GPS;           // wave loads per side and stage
    constexpr int LPW = 2 * LPS / NW;           // wave loads per wave and stage
    // [buffer][side][slice][column][slot] of 16-byte pieces
    __shared__ __attribute__((aligned(16))) uint4 sbuf[2][2][NSLICE][T][4];
    __shared__ int64_t s_pre[FIND_LDS_MAX + 1];
    const int64_t b = blockIdx.x;
    const int f = find_frag_lds(pre, nfrag, b, s_pre);
    const FragDev &F = fr[f];
    const int N = F.N;
    const int nt = (N + T - 1) / T;
    const int npairs = nt * (nt + 1) / 2;
    const int64_t lb = b - (nfrag <= FIND_LDS_MAX ? s_pre[f] : pre[f]);
    const int w = (int)(lb / npairs), pair = (int)(lb - (int64_t)w * npairs);
    int tp, tq;
    tri_decode(pair, tp, tq);
    const int p0 = tp * T, q0 = tq * T;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int wi = wave / WJN, wj = wave % WJN;   // 64-row block, 32-col block

    const int64_t Kp = F.Kpad8;
    const int8_t *slw = F.sl8 + (int64_t)w * NSLICE * N * Kp;

    v4i_t L0[4][2], L1[4][2], L2[4][2], L3[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) L0[i][j] = L1[i][j] = L2[i][j] = L3[i][j] = (v4i_t){0, 0, 0, 0};

    // This wave's LPW wave loads of a stage: load id = LPW*wave + t -> side =
    // id/LPS, slice = (id%LPS)/GPS, column group = id%GPS.  Columns past N are
    // clamped to N-1: they only feed outputs that are never written.
    const int lcol = lane >> 2;
    const int lpiece = (lane & 3) ^ ((lane >> 4) & 3);
    int64_t goff[LPW];
#pragma unroll
    for (int t = 0; t < LPW; ++t) {
        const int id = LPW * wave + t;
        const int side = id / LPS, sl = (id % LPS) / GPS, g = id % GPS;
        int P = (side ? q0 : p0) + 16 * g + lcol;
        P = P < N ? P : N - 1;
        goff[t] = (int64_t)sl * N * Kp + (int64_t)P * KS8 + 16 * lpiece;
    }
    auto issue = [&](int buf, int k0) {
#pragma unroll
        for (int t = 0; t < LPW; ++t) {
            const int id = LPW * wave + t;
            const int side = id / LPS, sl = (id % LPS) / GPS, g = id % GPS;
            __builtin_amdgcn_global_load_lds((const void *)(slw + goff[t] + (int64_t)k0 * N),
                                             (lds_void_t *)&sbuf[buf][side][sl][16 * g][0], 16, 0, 0);
        }
    };
    auto frag = [&](int buf, int side, int s, int row) {
        const int cl = row & 15;
        const uint4 v = sbuf[buf][side][s][row][swz8(cl, lane >> 4)];
        return __builtin_bit_cast(v4i_t, v);
    };
#define MFMA8(a, b, c) c = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0)

    const int nst = (int)(Kp / KS8);
    issue(0, 0);
    for (int st = 0; st < nst; ++st) {
        const int buf = st & 1;
        __builtin_amdgcn_s_waitcnt(0);
        __syncthreads();   // stage st in sbuf[buf]; everyone is done with sbuf[buf^1]
        if (st + 1 < nst) issue(buf ^ 1, (st + 1) * KS8);
        v4i_t bq[NSLICE][2];
#pragma unroll
        for (int s2 = 0; s2 < NSLICE; ++s2)
#pragma unroll
            for (int j = 0; j < 2; ++j) bq[s2][j] = frag(buf, 1, s2, 32 * wj + 16 * j + (lane & 15));
#pragma unroll
        for (int ih = 0; ih < 4; ih += 2) {
            v4i_t a[2];
#pragma unroll
            for (int ii = 0; ii < 2; ++ii) a[ii] = frag(buf, 0, 0, 64 * wi + 16 * (ih + ii) + (lane & 15));
#pragma unroll
            for (int ii = 0; ii < 2; ++ii)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    MFMA8(a[ii], bq[0][j], L0[ih + ii][j]);
                    MFMA8(a[ii], bq[1][j], L1[ih + ii][j]);
                    MFMA8(a[ii], bq[2][j], L2[ih + ii][j]);
                    MFMA8(a[ii], bq[3][j], L3[ih + ii][j]);
                }
#pragma unroll
            for (int ii = 0; ii < 2; ++ii) a[ii] = frag(buf, 0, 1, 64 * wi + 16 * (ih + ii) + (lane & 15));
#pragma unroll
            for (int ii = 0; ii < 2; ++ii)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    MFMA8(a[ii], bq[0][j], L1[ih + ii][j]);
                    MFMA8(a[ii], bq[1][j], L2[ih + ii][j]);
                    MFMA8(a[ii], bq[2][j], L3[ih + ii][j]);
                }
#pragma unroll
            for (int ii = 0; ii < 2; ++ii) a[ii] = frag(buf, 0, 2, 64 * wi + 16 * (ih + ii) + (lane & 15));
#pragma unroll
            for (int ii = 0; ii < 2; ++ii)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    MFMA8(a[ii], bq[0][j], L2[ih + ii][j]);
                    MFMA8(a[ii], bq[1][j], L3[ih + ii][j]);
                }
#pragma unroll
            for (int ii = 0; ii < 2; ++ii) a[ii] = frag(buf, 0, 3, 64 * wi + 16 * (ih + ii) + (lane & 15));
#pragma unroll
            for (int ii = 0; ii < 2; ++ii)
#pragma unroll
                for (int j = 0; j < 2; ++j) MFMA8(a[ii], bq[0][j], L3[ih + ii][j]);
        }
    }
#undef MFMA8

    const double *scw = F.scale8 + (int64_t)w * N;
    double *C = F.Pi + (int64_t)w * N * N;
    const double c1 = 1.0 / 128.0, c2 = c1 * c1, c3 = c2 * c1;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int q = q0 + 32 * wj + 16 * j + (lane & 15);
            const double sq = q < N ? scw[q] : 0.0;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int p = p0 + 64 * wi + 16 * i + 4 * (lane >> 4) + r;
                if (p < N && q <= p) {
                    const double v = (double)L0[i][j][r] + c1 * (double)L1[i][j][r] +
                                     c2 * (double)L2[i][j][r] + c3 * (double)L3[i][j][r];
                    C[(int64_t)p * N + q] = v * (scw[p] * sq);
                }
            }
        }
}

// The 128x128 form: eight waves of 64x32, two stages of 64 k in LDS (one work-group
// per CU, two waves per SIMD).  Of a stage's 80 MFMAs per wave, the 32 of slice 0 of
// the p side run first, while the wave reads the other three p slices; the
// barrier follows, since the stage's buffer has then been read by every wave, and the
// loads of the stage after the next go into it.  The other 48 MFMAs cover those loads
// and the reads of the next stage's first operands.  A wave above the diagonal of a
// diagonal tile only stages.
//
// xcd: chunks of 32 consecutive tiles (which share panels) go to one XCD at a time,
// so that its CUs find each other's panels in their L2, and the XCDs stay balanced
// over fragments of different K (one contiguous range of the grid per XCD did not: 1.4
// times slower on the batch).
//
// At K = 10800, N = 1800, 24 frequencies 3.80 ms (221 TFLOP/s FP64-equivalent): 2.7 POP/s
// counting whole tiles, whose area is 1.21 times N (N + 1) / 2 there, of the 3.8 that the
// MFMAs allow at the clock of this load (1.8 GHz); the LDS reads (24 KB per wave and stage)
// come next.  Before: 4.19 ms with both stages in one array, where the compiler made the
// first read after the loads wait for them, 4.43 without xcd, 5.97 with one LDS read or
// wait ahead of each group of MFMAs.  32 fragments of the batch shapes: 14.7 ms (16.5,
// 17.5, 23.8).  Loads of later stages into L2 ahead of their use made it no faster.
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_syrk_i8_128(
    const FragDev *__restrict__ fr, const int64_t *__restrict__ pre, int nfrag, int xcd) {
    constexpr int T = 128;
    // [side][slice][column][slot] of 16-byte pieces.  Two arrays and not one with an
    // index: the compiler then knows that a read of one does not wait for the loads into the
    // other.
    __shared__ __attribute__((aligned(16))) uint4 sb0[2][NSLICE][T][4], sb1[2][NSLICE][T][4];
    __shared__ int64_t s_pre[FIND_LDS_MAX + 1];
    const int64_t b = xcd ? xcd_chunks(blockIdx.x, gridDim.x) : (int64_t)blockIdx.x;
    const int f = find_frag_lds(pre, nfrag, b, s_pre);
    const FragDev &F = fr[f];
    const int N = F.N;
    const int nt = (N + T - 1) / T;
    const int npairs = nt * (nt + 1) / 2;
    const int64_t lb = b - (nfrag <= FIND_LDS_MAX ? s_pre[f] : pre[f]);
    const int w = __builtin_amdgcn_readfirstlane((int)(lb / npairs));
    const int pair = (int)(lb - (int64_t)w * npairs);
    int tp, tq;
    tri_decode(pair, tp, tq);
    const int p0 = __builtin_amdgcn_readfirstlane(tp * T), q0 = __builtin_amdgcn_readfirstlane(tq * T);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int wi = wave >> 2, wj = wave & 3;   // 64x32 block of the tile
    const int64_t Kp = F.Kpad8;
    const int8_t *slw = F.sl8 + (int64_t)w * NSLICE * N * Kp;

    // A wave loads one slice of one side: 8 groups of 16 columns (1 KB per load; lane
    // l lands in column l/4, slot l%4).  Columns past N are whatever follows (the
    // allocation ends with SL_PAD spare bytes): they only feed outputs that are never
    // written.
    const int side = wave >> 2, slice = wave & 3;
    const int lpiece = (lane & 3) ^ ((lane >> 4) & 3);
    const uint32_t goff = (uint32_t)((side ? q0 : p0) + (lane >> 2)) * KS8 + 16u * lpiece;
    const char *base = (const char *)(slw + (int64_t)slice * N * Kp);
    auto issue = [&](int buf, int st) {
#if defined(__HIP_DEVICE_COMPILE__)
        typedef __attribute__((address_space(1))) const char gchar_t;
        // the load's constant offset counts for both addresses: four groups per base
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const char *src = base + ((int64_t)st * KS8 * N + 64 * KS8 * h);
            asm("" : "+s"(src));   // a scalar base, the lane's offset in 32 bits
            auto *from = (const __attribute__((address_space(1))) void *)((gchar_t *)src + goff);
            auto *to = (lds_void_t *)(buf ? &sb1[side][slice][64 * h][0] : &sb0[side][slice][64 * h][0]);
            __builtin_amdgcn_global_load_lds(from, to, 16, 0, 0);
            __builtin_amdgcn_global_load_lds(from, to, 16, 1024, 0);
            __builtin_amdgcn_global_load_lds(from, to, 16, 2048, 0);
            __builtin_amdgcn_global_load_lds(from, to, 16, 3072, 0);
        }
#endif
    };
    const int nst = (int)(Kp / KS8);
    issue(0, 0);
    if (tp == tq && 32 * wj > 64 * wi + 63) {
        __syncthreads();
        if (nst > 1) issue(1, 1);
        for (int st = 0; st < nst; ++st) {
            __syncthreads();
            issue(st & 1, min(st + 2, nst - 1));
        }
        __builtin_amdgcn_s_waitcnt(0);
        return;
    }
    // slice s of the wave's 16-column groups of the p side (four) and the q side (two)
    const int fo = (lane & 15) * 4 + swz8(lane & 15, lane >> 4);
    auto fragp = [&](v4i_t (&v)[4], int buf, int s) {
        const uint4 *L = buf ? &sb1[0][s][64 * wi][0] : &sb0[0][s][64 * wi][0];
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = __builtin_bit_cast(v4i_t, L[64 * i + fo]);
    };
    auto fragq = [&](v4i_t (&v)[2], int buf, int s) {
        const uint4 *L = buf ? &sb1[1][s][32 * wj][0] : &sb0[1][s][32 * wj][0];
#pragma unroll
        for (int j = 0; j < 2; ++j) v[j] = __builtin_bit_cast(v4i_t, L[64 * j + fo]);
    };
    v4i_t L0[4][2], L1[4][2], L2[4][2], L3[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) L0[i][j] = L1[i][j] = L2[i][j] = L3[i][j] = (v4i_t){0, 0, 0, 0};
    auto mma = [&](const v4i_t (&a)[4], const v4i_t (&b)[2], v4i_t (&c)[4][2]) {
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
                c[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[i], b[j], c[i][j], 0, 0, 0);
    };
    v4i_t a0[4], a1[4], a2[4], a3[4], b0[2], b1[2], b2[2], b3[2];
    __syncthreads();
    if (nst > 1) issue(1, 1);
    fragp(a0, 0, 0);
    fragq(b0, 0, 0);
    fragq(b1, 0, 1);
    fragq(b2, 0, 2);
    fragq(b3, 0, 3);
    // the last stages load and read stage nst - 1 again, unused
    auto stage = [&](int buf, int st) {
        fragp(a1, buf, 1);
        fragp(a2, buf, 2);
        fragp(a3, buf, 3);
        mma(a0, b3, L3);
        mma(a0, b2, L2);
        mma(a0, b1, L1);
        mma(a0, b0, L0);
#pragma unroll
        for (int u = 0; u < 12; ++u) {
            __builtin_amdgcn_sched_group_barrier(0x8, 2, 0);     // MFMA
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // LDS read
        }
        __builtin_amdgcn_sched_group_barrier(0x8, 8, 0);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        issue(buf, min(st + 2, nst - 1));
        mma(a1, b2, L3);
        mma(a1, b1, L2);
        mma(a1, b0, L1);
        mma(a2, b1, L3);
        mma(a2, b0, L2);
        mma(a3, b0, L3);
        fragq(b3, buf ^ 1, 3);
        fragp(a0, buf ^ 1, 0);
        fragq(b2, buf ^ 1, 2);
        fragq(b1, buf ^ 1, 1);
        fragq(b0, buf ^ 1, 0);
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            __builtin_amdgcn_sched_group_barrier(0x8, 2, 1);
            __builtin_amdgcn_sched_group_barrier(0x20, 1, 1);    // global -> LDS
        }
#pragma unroll
        for (int u = 0; u < 10; ++u) {
            __builtin_amdgcn_sched_group_barrier(0x8, 3, 1);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
        }
        __builtin_amdgcn_sched_group_barrier(0x8, 2, 1);
        __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
        __builtin_amdgcn_sched_barrier(0);
    };
    for (int st = 0; st < nst; st += 2) {   // Kpad8 is a multiple of 128: an even number
        stage(0, st);
        stage(1, st + 1);
    }
    __builtin_amdgcn_s_waitcnt(0);   // no load into LDS outlives the work-group

    const double *scw = F.scale8 + (int64_t)w * N;
    double *C = F.Pi + (int64_t)w * N * N;
    const double c1 = 1.0 / 128.0, c2 = c1 * c1, c3 = c2 * c1;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        double sp[4];
#pragma unroll
        for (int r = 0; r < 4; ++r)
            sp[r] = scw[min(p0 + 64 * wi + 16 * i + 4 * (lane >> 4) + r, N - 1)];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int q = q0 + 32 * wj + 16 * j + (lane & 15);
            const double sq = scw[min(q, N - 1)];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int p = p0 + 64 * wi + 16 * i + 4 * (lane >> 4) + r;
                const double v = (double)L0[i][j][r] + c1 * (double)L1[i][j][r] +
                                 c2 * (double)L2[i][j][r] + c3 * (double)L3[i][j][r];
                if (p < N && q <= p) C[(int64_t)p * N + q] = v * (sp[r] * sq);
            }
        }
    }
}

int syrk_i8_tile(int variant) { return variant == I8V_T64 ? 64 : 128; }

int launch_syrk_i8(brpa_ctx *ctx, const FragDev *fr, const int64_t *pre, int nfrag, int64_t total,
                   int variant) {
    if (total <= 0) return BRPA_OK;
    switch (variant) {
    case I8V_T128:
        hipLaunchKernelGGL(k_syrk_i8_128, dim3((unsigned)total), dim3(512), 0, ctx->stream, fr,
                           pre, nfrag, 0);
        break;
    case I8V_T128_XCD:
        hipLaunchKernelGGL(k_syrk_i8_128, dim3((unsigned)total), dim3(512), 0, ctx->stream, fr,
                           pre, nfrag, 1);
        break;
    case I8V_T64:
        hipLaunchKernelGGL(k_syrk_i8_64, dim3((unsigned)total), dim3(128), 0, ctx->stream, fr,
                           pre, nfrag);
        break;
    default:
        return brpa_fail(ctx, BRPA_ERR_ARG, "unknown split-int8 kernel variant %d", variant);
    }
    LAUNCH_CHECK(ctx);
    return BRPA_OK;
}
