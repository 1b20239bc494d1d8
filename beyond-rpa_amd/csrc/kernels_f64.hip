// FP64 kernels of the E_RPA hot path on gfx950 (CDNA4).
//
//   k_dtab         c_w(ai) = 4 d/(d^2+u_w^2)           (rpa_core_MO.f90:379-401)
//   k_syrk_f64     Pi_w = R^T diag(c_w) R on v_mfma_f64_16x16x4_f64, one R tile in
//                  LDS shared by 4 waves = 4 frequencies, or the quadrants of one
//                  frequency's tile  (dgemm of rpa_core_MO.f90:402)
//   k_set_diag     diag_w (tr Pi, rpa_CC.f90:444-447); Pi_w[P][P] += 1 (448-450)
//   k_potrf_diag   Cholesky + inverse of a 64x64 diagonal block (four waves)
//   k_chol_panel   left-looking update of a 64-column strip and L21 = B L11^{-T}
//   k_chol_rest    rank-256 update of the rest of the trailing matrix
//   k_chol_step    diagonal block, left-looking strip and L21 of a step in one launch
//   k_energy       E = sum_w w/(2 pi) (2 sum log L_kk - tr Pi_w)  (rpa_CC.f90:451-453)
//
// All kernels walk a flattened work list over fragments: work-group b belongs
// to fragment f with pre[f] <= b < pre[f+1].
#include "gemm_tile.h"
#include "internal.h"

#define LAUNCH_CHECK(ctx)                                                                      \
    do {                                                                                       \
        hipError_t _e = hipGetLastError();                                                     \
        if (_e != hipSuccess)                                                                  \
            return brpa_fail((ctx), BRPA_ERR_HIP, "kernel launch failed: %s (%s:%d)",          \
                             hipGetErrorString(_e), __FILE__, __LINE__);                       \
    } while (0)

static inline unsigned grid1(int64_t total) { return (unsigned)total; }

typedef double d2v_t __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(1))) const double gdouble_t;
typedef __attribute__((address_space(1))) double gdouble_mut_t;

// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_dtab(const FragDev *__restrict__ fr,
                                             const int64_t *__restrict__ pre, int nfrag) {
    int64_t b = blockIdx.x;
    int f = find_frag(pre, nfrag, b);
    const FragDev &F = fr[f];
    int64_t e = (b - pre[f]) * 256 + threadIdx.x;
    int64_t tot = (int64_t)F.F * F.K;
    if (e >= tot) return;
    int w = (int)(e / F.K);
    int k = (int)(e - (int64_t)w * F.K);
    int i = k / F.nvir, a = k - i * F.nvir;
    double d = F.evir[a] - F.eocc[i];
    double u = F.freqs[w];
    const double c = 4.0 * d / (d * d + u * u);
    const_cast<double *>(F.dtab)[e] = c;
    if (F.sdtab) const_cast<double *>(F.sdtab)[e] = sqrt(c);
}

int launch_dtab(brpa_ctx *ctx, const FragDev *fr, const int64_t *pre, int nfrag, int64_t total) {
    if (total <= 0) return BRPA_OK;
    hipLaunchKernelGGL(k_dtab, dim3(grid1(total)), dim3(256), 0, ctx->stream, fr, pre, nfrag);
    LAUNCH_CHECK(ctx);
    return BRPA_OK;
}

// ---------------------------------------------------------------------------
// FP64 SYRK on MFMA: one 64x64 tile pair (tp >= tq) per work-group, the two 64-column
// panels of R staged in LDS 16 rows at a time.
//
// MFMA v_mfma_f64_16x16x4_f64 operand layout (lane l):
//   A[m = l%16][k = l/16], B[k = l/16][n = l%16],
//   D: 4 doubles, D[r] = C[m = l/16 + 4*r][n = l%16]  (probed on gfx950; the
//   f32 shapes use 4*(l/16) + r instead).
// Step s (of 4) of a stage takes the rows 4 s + l/16.
//
//   wide  (QUAD = false)  four frequencies per work-group: wave w computes the whole
//         tile for frequency 4 g + w, so R is staged once for four products
//   quad  (QUAD = true)   one frequency: wave (w/2, w%2) computes a 32x32 quadrant,
//         for launches whose wide form would not fill the chip (syrk_quad)
//
// The stages go straight from global memory into LDS (16 bytes per lane), double-buffered,
// rows of 64 doubles with the 16-double blocks of odd rows swapped in pairs, so that the
// four lane groups of an operand read (four consecutive rows) hit both halves of the 64
// banks.  Columns past N repeat the last pair: they only reach products that are not
// stored.  A last stage with fewer than 16 rows, or one whose loads would end past R,
// goes through registers with zeros past K.  A diagonal tile needs one panel and the
// blocks i >= j only.
//
// Bound by MFMA issue.  The reads of one half of a stage run while the other half is
// multiplied, the barrier stands between the halves (as in k_gemm_f64).  Measured at
// K = 19200, N = 2400, 16 frequencies: 64.9 TFLOP/s (56.2 with register-staged
// stages between two barriers).  A batch of 12 fragments, half of them with odd N: 23.9
// ms with four bytes per lane for those, 23.4.
constexpr int KB = 16;                    // rows of R per LDS stage
constexpr int SYRK_P = KB * SYRK_T;       // doubles per panel stage

struct SyrkPanel {
    uint32_t off[2];   // the two loads of a wave
};

// byte offsets from R + k0 N + c0 of the lane's part of a wave's loads
__device__ __forceinline__ SyrkPanel syrk_panel(int N, int c0, int wave, int lane) {
    SyrkPanel p;
#pragma unroll
    for (int t = 0; t < 2; ++t) {
        const int kr = 4 * wave + 2 * t + (lane >> 5);
        const int c = 2 * ((lane & 31) ^ (8 * (kr & 1)));
        p.off[t] = 8u * ((uint32_t)kr * (uint32_t)N + (uint32_t)(min(c0 + c, (N - 1) & ~1) - c0));
    }
    return p;
}

__device__ __forceinline__ void syrk_stage(const SyrkPanel &p, const char *base, double *L, int wave) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef __attribute__((address_space(1))) const char gchar_t;
    typedef __attribute__((address_space(3))) void lvoid_t;
#pragma unroll
    for (int t = 0; t < 2; ++t)
        __builtin_amdgcn_global_load_lds(
            (const __attribute__((address_space(1))) void *)((gchar_t *)base + p.off[t]),
            (lvoid_t *)(L + (4 * wave + 2 * t) * SYRK_T), 16, 0, 0);
#endif
}
__device__ __forceinline__ void syrk_stage_tail(const double *__restrict__ R, int K, int N, int k0,
                                                int c0, double *L, int tid) {
    const gdouble_t *G = (const gdouble_t *)R;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int kr = (tid >> 6) + 4 * u, c = tid & 63;
        const bool ok = k0 + kr < K && c0 + c < N;
        const double v = G[ok ? (int64_t)(k0 + kr) * N + c0 + c : 0];
        L[kr * SYRK_T + (c ^ (16 * (kr & 1)))] = ok ? v : 0.0;
    }
}

template <bool QUAD, bool DIAG>
__device__ __forceinline__ void syrk_f64_tile(const FragDev &F, int w0, int tp, int tq, int both,
                                              double *__restrict__ sA0, double *__restrict__ sA1,
                                              double *__restrict__ sB0, double *__restrict__ sB1) {
    const double *__restrict__ R = F.R;
    const int K = F.K, N = F.N;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int p0 = tp * SYRK_T, q0 = tq * SYRK_T;
    const int w = QUAD ? w0 : w0 + wave;
    constexpr int NB = QUAD ? 2 : 4;            // 16-row blocks per wave and side
    const int bi = QUAD ? 2 * (wave >> 1) : 0, bj = QUAD ? 2 * (wave & 1) : 0;
    // waves past the last frequency, and the quadrant above the diagonal, only stage
    const bool active = w < F.F && !(QUAD && DIAG && bj > bi);
    const int rl = lane & 15, g4 = lane >> 4;
    const SyrkPanel pa = syrk_panel(N, p0, wave, lane);
    const SyrkPanel pb = DIAG ? pa : syrk_panel(N, q0, wave, lane);
    const char *ba = reinterpret_cast<const char *>(R + p0);
    const char *bb = reinterpret_cast<const char *>(R + q0);
    // with an odd N the last column's pair of row K - 1 would end past R
    const bool over = (N & 1) && p0 + SYRK_T > N;
    const int nfull = (K - (over ? 1 : 0)) / KB, ns = (K + KB - 1) / KB;
    auto stage = [&](int buf, int q) {
        const int64_t o = 8 * (int64_t)N * (KB * q);
        syrk_stage(pa, ba + o, buf ? sA1 : sA0, wave);
        if (!DIAG) syrk_stage(pb, bb + o, buf ? sB1 : sB0, wave);
    };
    auto put = [&](int buf, int q) {
        if (q < nfull) {
            stage(buf, q);
        } else if (q < ns) {
            syrk_stage_tail(R, K, N, KB * q, p0, buf ? sA1 : sA0, tid);
            if (!DIAG) syrk_stage_tail(R, K, N, KB * q, q0, buf ? sB1 : sB0, tid);
        }
    };
    put(0, 0);
    if (!active) {
        __syncthreads();
        put(1, 1);
        for (int q = 0; q + 1 < ns; ++q) {
            __syncthreads();
            put(q & 1, q + 2);
        }
        return;
    }
    d4_t acc[NB][NB];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = (d4_t){0.0, 0.0, 0.0, 0.0};
    // element (row 4 s + g4, column 16 b + rl) of a stage; the block index of odd rows
    // has its low bit flipped
    const int x0 = g4 * SYRK_T + rl + 16 * (g4 & 1), x1 = g4 * SYRK_T + rl - 16 * (g4 & 1);
    auto frags = [&](double (&a)[2][NB], double (&b)[2][NB], int buf, int h) {
        const double *LA = (buf ? sA1 : sA0) + 16 * bi;
        const double *LB = (DIAG ? (buf ? sA1 : sA0) : (buf ? sB1 : sB0)) + 16 * bj;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
#pragma unroll
            for (int i = 0; i < NB; ++i)
                a[s][i] = LA[(i & 1 ? x1 : x0) + 16 * i + 4 * (2 * h + s) * SYRK_T];
#pragma unroll
            for (int j = 0; j < NB; ++j)
                b[s][j] = LB[(j & 1 ? x1 : x0) + 16 * j + 4 * (2 * h + s) * SYRK_T];
        }
    };
    auto mma = [&](const double (&a)[2][NB], const double (&b)[2][NB], double d0, double d1) {
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const double x = a[s][i] * (s ? d1 : d0);
#pragma unroll
                for (int j = 0; j < NB; ++j)
                    if (QUAD || !DIAG || i >= j)
                        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(x, b[s][j], acc[i][j], 0, 0, 0);
            }
    };
    // c_w of the lane's rows of stage q: two for either half
    const gdouble_t *dt = (const gdouble_t *)F.dtab + (int64_t)w * K;
    auto coef = [&](double (&d)[4], int q, int h) {
#pragma unroll
        for (int s = 2 * h; s < 2 * h + 2; ++s) {
            const int k = KB * q + 4 * s + g4;
            d[s] = dt[min(k, K - 1)];   // rows past K are zero
        }
    };
    double a0[2][NB], b0[2][NB], a1[2][NB], b1[2][NB], de[4], dd[4];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        coef(de, 0, h);
        coef(dd, min(1, ns - 1), h);
    }
    __syncthreads();
    put(1, 1);
    frags(a0, b0, 0, 0);
    // buf constant, arrays of their own: as in gemm_tile.h.  d: c_w of this stage, replaced by
    // that of the stage after the next as soon as it is used; loaded one stage ahead, just before
    // the barrier that waits for it, it held up the quad form at every stage (840 work-groups
    // of 517 rows: 97 us instead of 86).
    auto step = [&](int buf, int q, double (&d)[4]) {
        frags(a1, b1, buf, 1);
        mma(a0, b0, d[0], d[1]);
        constexpr int NM = QUAD ? 8 : (DIAG ? 20 : 32), NR = QUAD ? 4 : 8;
#pragma unroll
        for (int u = 0; u < NR; ++u) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);     // MFMA
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // LDS read
        }
        __builtin_amdgcn_sched_group_barrier(0x8, NM - NR, 0);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        frags(a0, b0, buf ^ 1, 0);
        coef(d, q + 2, 0);
        stage(buf, q + 2);
        mma(a1, b1, d[2], d[3]);
        constexpr int NL = 2 + 2 * (DIAG ? 1 : 2);
        constexpr int NL1 = NL < NM - NR ? NL : NM - NR;
#pragma unroll
        for (int u = 0; u < NR; ++u) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 1);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
        }
#pragma unroll
        for (int u = 0; u < NL1; ++u) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 1);
            __builtin_amdgcn_sched_group_barrier(0x20, (NL + NL1 - 1) / NL1, 1);   // global loads
        }
        __builtin_amdgcn_sched_group_barrier(0x8, NM - NR - NL1, 1);
        __builtin_amdgcn_sched_barrier(0);
        coef(d, q + 2, 1);
    };
    int q = 0;
    for (; q + 3 < nfull; q += 2) {
        step(0, q, de);
        step(1, q + 1, dd);
    }
    int buf = 0;
    for (; q < ns; ++q, buf ^= 1) {
        frags(a1, b1, buf, 1);
        mma(a0, b0, de[0], de[1]);
        if (q + 1 < ns) {
            __syncthreads();
            put(buf, q + 2);
            frags(a0, b0, buf ^ 1, 0);
        }
        mma(a1, b1, de[2], de[3]);
#pragma unroll
        for (int s = 0; s < 4; ++s) de[s] = dd[s];
#pragma unroll
        for (int h = 0; h < 2; ++h) coef(dd, min(q + 2, ns - 1), h);
    }

    gdouble_mut_t *C = (gdouble_mut_t *)(F.Pi + (int64_t)w * N * N);
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) {
            if (DIAG && bi + i < bj + j) continue;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int p = p0 + 16 * (bi + i) + g4 + 4 * r;
                const int c = q0 + 16 * (bj + j) + rl;
                if (p < N && c <= p) {
                    const double v = acc[i][j][r];
                    C[(int64_t)p * N + c] = v;
                    if (both) C[(int64_t)c * N + p] = v;
                }
            }
        }
}

// Work-groups per fragment: syrk_items(N, F, QUAD), pair-major within a frequency
// (group).  both: the upper triangle of Pi is written too.
template <bool QUAD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, QUAD ? 4 : 2))) void
k_syrk_f64(const FragDev *__restrict__ fr, const int64_t *__restrict__ pre, int nfrag, int both) {
    __shared__ __attribute__((aligned(16))) double sA0[SYRK_P], sA1[SYRK_P], sB0[SYRK_P], sB1[SYRK_P];
    int64_t b = blockIdx.x;
    int f = find_frag(pre, nfrag, b);
    const FragDev &F = fr[f];
    int64_t lb = b - pre[f];
    int nt = (F.N + SYRK_T - 1) / SYRK_T;
    int npairs = nt * (nt + 1) / 2;
    int g = (int)(lb / npairs), pair = (int)(lb - (int64_t)g * npairs);
    int tp, tq;
    tri_decode(pair, tp, tq);
    const int w0 = QUAD ? g : 4 * g;
    if (tp == tq)
        syrk_f64_tile<QUAD, true>(F, w0, tp, tq, both, sA0, sA1, sB0, sB1);
    else
        syrk_f64_tile<QUAD, false>(F, w0, tp, tq, both, sA0, sA1, sB0, sB1);
}

int64_t syrk_items(int64_t N, int64_t F, bool quad) {
    const int64_t nt = (N + SYRK_T - 1) / SYRK_T;
    return nt * (nt + 1) / 2 * (quad ? F : (F + 3) / 4);
}

// In units of one tile's four products on a CU: the wide form takes one per
// work-group, the quad form a quarter, at 1.2 times the cost (twice the LDS reads and
// four times the loads per product).  What decides is the last round of work-groups
// over the CUs.  Measured (wide, quad, us): 112 tiles 84, 59; 220 tiles 401, 466;
// 360 tiles of 10 frequencies 897, 688, of 12 954, 928; 612 tiles 1803, 1829; 2610
// tiles 13794, 16927.
bool syrk_quad(const brpa_ctx *ctx, int64_t wide_total, int64_t quad_total) {
    const int64_t ncu = ctx->ncu > 0 ? ctx->ncu : 256;
    const int64_t wide = (wide_total + ncu - 1) / ncu, quad = (quad_total + ncu - 1) / ncu;
    return 0.25 * 1.2 * (double)quad < (double)wide;
}

int launch_syrk_f64(brpa_ctx *ctx, const FragDev *fr, const int64_t *pre, int nfrag, int64_t total,
                    bool quad, bool both) {
    if (total <= 0) return BRPA_OK;
    if (quad)
        hipLaunchKernelGGL(k_syrk_f64<true>, dim3(grid1(total)), dim3(256), 0, ctx->stream, fr, pre,
                           nfrag, both ? 1 : 0);
    else
        hipLaunchKernelGGL(k_syrk_f64<false>, dim3(grid1(total)), dim3(256), 0, ctx->stream, fr,
                           pre, nfrag, both ? 1 : 0);
    LAUNCH_CHECK(ctx);
    return BRPA_OK;
}

// 16 rows of a 64 x 64 tile pair per work-group: the sum of the partial tiles is added
// to P as it is and, off the diagonal, transposed through LDS.  Bound by memory:
// (nq / 2 + 2) N^2 doubles: 11 us at N = 905, nq = 4 and 7 (30 us with a whole tile pair
// per work-group at 7).
__global__ __launch_bounds__(256) void k_syrk_acc(double *__restrict__ P,
                                                 const double *__restrict__ S, int N, int nq) {
    __shared__ double sT[16][65];
    int ti, tj;
    tri_decode((int)blockIdx.x >> 2, ti, tj);
    const int c = threadIdx.x & 63, r0 = threadIdx.x >> 6;
    const int row0 = 64 * ti + 16 * ((int)blockIdx.x & 3), col = 64 * tj + c;
    const int64_t NN = (int64_t)N * N;
    double s[4] = {0.0, 0.0, 0.0, 0.0}, p[4] = {0.0, 0.0, 0.0, 0.0};
    int64_t e[4];
    bool ok[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = row0 + r0 + 4 * i;
        ok[i] = row < N && col <= row;
        e[i] = ok[i] ? (int64_t)row * N + col : 0;
        p[i] = P[e[i]];
    }
#pragma unroll 4
    for (int q = 0; q < nq; ++q)
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i] += S[q * NN + e[i]];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (ok[i]) P[e[i]] = p[i] + s[i];
        sT[r0 + 4 * i][c] = s[i];
    }
    __syncthreads();
    // rows of the transposed tile: 16 columns each
    const int tc = threadIdx.x & 15, tr = threadIdx.x >> 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int r = 64 * tj + tr + 16 * i, cc = row0 + tc;
        if (cc < N && r < cc) P[(int64_t)r * N + cc] += sT[tc][tr + 16 * i];
    }
}

int launch_syrk_acc(brpa_ctx *ctx, double *P, const double *S, int64_t N, int nq) {
    const int64_t nt = (N + 63) / 64;
    hipLaunchKernelGGL(k_syrk_acc, dim3(grid1(2 * nt * (nt + 1))), dim3(256), 0, ctx->stream, P, S,
                       (int)N, nq);
    LAUNCH_CHECK(ctx);
    return BRPA_OK;
}

// ---------------------------------------------------------------------------
// diag_w[P] and Pi_w[P][P] = diag_w[P] + 1.  The diagonal is either the one the
// FP64 SYRK (or the caller) computed, or, for the split-BF16 form, the exact
// double-double sum of the per-block partials written by k_split.
// Work-groups per fragment: ceil(F*N/256).
__global__ __launch_bounds__(256) void k_set_diag(const FragDev *__restrict__ fr,
                                                 const int64_t *__restrict__ pre, int nfrag,
                                                 int mode) {
    int64_t b = blockIdx.x;
    int f = find_frag(pre, nfrag, b);
    const FragDev &F = fr[f];
    int64_t e = (b - pre[f]) * 256 + threadIdx.x;
    if (e >= (int64_t)F.F * F.N) return;
    int w = (int)(e / F.N), P = (int)(e - (int64_t)w * F.N);
    double *pp = F.Pi + (int64_t)w * F.N * F.N + (int64_t)P * F.N + P;
    // mode 0: Pi's own diagonal; 1: sum of the split-BF16 double-double block
    // partials; 2: diag already holds the exact value (split-int8 column pass)
    double d;
    if (mode == 1) {
        dd_t s = {0.0, 0.0};
        for (int blk = 0; blk < F.nblk; ++blk) {
            const double *q = F.dpart + (((int64_t)w * F.nblk + blk) * F.N + P) * 2;
            s = dd_add(s, (dd_t){q[0], q[1]});
        }
        d = s.hi + s.lo;
    } else if (mode == 2) {
        d = F.diag[e];
    } else {
        d = *pp;
    }
    F.diag[e] = d;
    *pp = d + 1.0;
}

int launch_set_diag(brpa_ctx *ctx, const FragDev *fr, const int64_t *pre, int nfrag, int64_t total,
                    int mode) {
    if (total <= 0) return BRPA_OK;
    hipLaunchKernelGGL(k_set_diag, dim3(grid1(total)), dim3(256), 0, ctx->stream, fr, pre, nfrag,
                       mode);
    LAUNCH_CHECK(ctx);
    return BRPA_OK;
}

// ---------------------------------------------------------------------------
// Blocked Cholesky of A_w = 1 + Pi_w (lower triangle, row-major) in 64-column steps j
// (j0 = 64 j), one launch per step for few matrices (k_chol_step), else two:
//   k_potrf_diag   one work-group per matrix: factors the diagonal block in LDS,
//                  writes its log-det partial and L11^{-1} (own buffer; A11
//                  itself is never written back, so no work-group of the same
//                  step can read a half-factored block)
//   k_chol_panel   64 rows of the step's columns: the outer panel's earlier columns
//                  applied, then L21
// and after every outer panel of four steps k_chol_rest, the rest of A22 (launch_cholesky).
// Work-groups per fragment: chol_items.

// 1 / p for p within 2^-1000 .. 2^1000: the hardware estimate and two Newton
// steps (5 dependent instructions instead of the ~12 of a division)
__device__ __forceinline__ double rcp_newton(double p) {
    double x = __builtin_amdgcn_rcp(p);
    x = fma(fma(-p, x, 1.0), x, x);
    return fma(fma(-p, x, 1.0), x, x);
}

// Cholesky factor of a 64 x 64 block by one work-group of four waves.  The block sits in
// LDS as 4 x 4 blocks of 16 (lower triangle; the upper one is scratch):
//   panel p     wave 0: lane r holds row r of the 16 panel columns in registers
//               and eliminates column by column.  Beside it every row of 16 lanes holds
//               the 16 pivot rows, so that the row of the pivot comes by the
//               row_newbcast operand of the multiply-add itself (by readlane it took two
//               reads, a wait and the multiply-add), and neither LDS access nor square
//               root lies between two pivots; the columns are scaled by 1 / sqrt(pivot)
//               at the end, all 16 at once.
//   column p+1  waves 1-3: A(i, p+1) -= L(i, p) L(p+1, p)^T on MFMA
//   the other blocks right of it by waves 1-3 while wave 0 runs panel p+1, and after
//               them work(p + 1), the caller's own
//   L(p, p)^{-1}  from panel p itself, whose lanes 0 .. 15 would idle: rows of the
//               identity below the block become those of L(p, p)^{-T}.  Panel 0 has no
//               idle lanes; wave 2 inverts its block during panel 2.
// The block's own diagonal, 1 + Pi, stays apart (T.diag) and S starts with zeros there:
// the updates, small beside the 1, are summed by themselves and added to it once, when
// the pivot is due.  Added to it one by one they leave an error of 26 x 2^-53 in E(u) at
// N = 64, so 11; the addition costs 0.17 us a block (k_chol_step 28.2 us, 28.4 so).
// chol_panels returns whether a pivot was not positive.
//
// Bound by latency: 64 pivots in a chain of broadcast, reciprocal, multiply and
// multiply-add.  Measured on MI355X: 21700 cycles for the four panels (26600 by
// readlane); a k_potrf_diag launch of 160 matrices 15 us (17.7; 61.3 for one left-looking
// wave per matrix with rows of L from LDS, the square root and division in the chain
// and the whole inverse by substitution).
constexpr int CH_LP = CHOL_NB + 2;   // row pitch: 16-byte aligned rows, 16 rows on 16 distinct 4-bank groups
constexpr int CH_XP = 18;

struct CholLds {
    double S[CHOL_NB][CH_LP];
    double Xd[4][16][CH_XP];   // L(p, p)^{-1}
    double rdiag[CHOL_NB];
    double diag[CHOL_NB];      // of the given block
};

// the block at (j0, j0): lower triangle only; rows and columns past nbj are those of
// the identity
__device__ __forceinline__ void chol_load64(CholLds &T, const gdouble_t *G, int N, int j0, int nbj,
                                            int wave, int lane) {
    double v[16];
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int r = wave + 4 * u;
        const bool in = r < nbj && lane <= r;
        v[u] = G[in ? (int64_t)(j0 + r) * N + j0 + lane : 0];
        v[u] = in ? v[u] : ((r >= nbj && lane == r) ? 1.0 : 0.0);
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) {
        const int r = wave + 4 * u;
        T.S[r][lane] = lane == r ? 0.0 : v[u];
        if (lane == r) T.diag[r] = v[u];
    }
}

// L(p, p)^{-1} by substitution (lane n: column n): x_i = (delta_in - sum_{k<i} L_ik x_k) / L_ii
__device__ __forceinline__ void chol_invert16(CholLds &T, int p, int lane) {
    const int l16 = lane & 15;
    double x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        double s0 = i == l16 ? 1.0 : 0.0, s1 = 0.0;
#pragma unroll
        for (int k = 0; k < i; k += 2) {
            const d2v_t u = *reinterpret_cast<const d2v_t *>(&T.S[16 * p + i][16 * p + k]);
            s0 = fma(-u.x, x[k], s0);
            if (k + 1 < i) s1 = fma(-u.y, x[k + 1], s1);
        }
        x[i] = (s0 + s1) * T.rdiag[16 * p + i];
    }
    if (lane < 16)
#pragma unroll
        for (int i = 0; i < 16; ++i) T.Xd[p][i][l16] = x[i];
}

// x + y * (v of lane j of the lane's row of 16), for columns J .. J + n - 1 of the pivot
// rows d and of the lane's own row a.  The s_nop keeps the two wait states between a
// vector write of dc and its cross-lane read.
#define CHOL_DPP(x, y, j) \
    "v_fmac_f64_dpp %[" x "], %[dc], %[" y "] row_newbcast:%[" j "] row_mask:0xf bank_mask:0xf\n\t"
template <int J, int NJ>
__device__ __forceinline__ void chol_eliminate(double (&d)[16], double (&a)[16], double dc, double md,
                                               double ma) {
#if defined(__HIP_DEVICE_COMPILE__)
    if constexpr (NJ >= 5) {
        asm("s_nop 1\n\t"
            CHOL_DPP("d0", "md", "j0") CHOL_DPP("a0", "ma", "j0")
            CHOL_DPP("d1", "md", "j1") CHOL_DPP("a1", "ma", "j1")
            CHOL_DPP("d2", "md", "j2") CHOL_DPP("a2", "ma", "j2")
            CHOL_DPP("d3", "md", "j3") CHOL_DPP("a3", "ma", "j3")
            CHOL_DPP("d4", "md", "j4") CHOL_DPP("a4", "ma", "j4")
            : [d0] "+&v"(d[J + 0]), [a0] "+&v"(a[J + 0]), [d1] "+&v"(d[J + 1]), [a1] "+&v"(a[J + 1]), [d2] "+&v"(d[J + 2]), [a2] "+&v"(a[J + 2]), [d3] "+&v"(d[J + 3]), [a3] "+&v"(a[J + 3]), [d4] "+&v"(d[J + 4]), [a4] "+&v"(a[J + 4])
            : [dc] "v"(dc), [md] "v"(md), [ma] "v"(ma), [j0] "n"(J + 0), [j1] "n"(J + 1), [j2] "n"(J + 2), [j3] "n"(J + 3), [j4] "n"(J + 4));
        chol_eliminate<J + 5, NJ - 5>(d, a, dc, md, ma);
    } else if constexpr (NJ == 4) {
        asm("s_nop 1\n\t"
            CHOL_DPP("d0", "md", "j0") CHOL_DPP("a0", "ma", "j0")
            CHOL_DPP("d1", "md", "j1") CHOL_DPP("a1", "ma", "j1")
            CHOL_DPP("d2", "md", "j2") CHOL_DPP("a2", "ma", "j2")
            CHOL_DPP("d3", "md", "j3") CHOL_DPP("a3", "ma", "j3")
            : [d0] "+&v"(d[J + 0]), [a0] "+&v"(a[J + 0]), [d1] "+&v"(d[J + 1]), [a1] "+&v"(a[J + 1]), [d2] "+&v"(d[J + 2]), [a2] "+&v"(a[J + 2]), [d3] "+&v"(d[J + 3]), [a3] "+&v"(a[J + 3])
            : [dc] "v"(dc), [md] "v"(md), [ma] "v"(ma), [j0] "n"(J + 0), [j1] "n"(J + 1), [j2] "n"(J + 2), [j3] "n"(J + 3));
    } else if constexpr (NJ == 3) {
        asm("s_nop 1\n\t"
            CHOL_DPP("d0", "md", "j0") CHOL_DPP("a0", "ma", "j0")
            CHOL_DPP("d1", "md", "j1") CHOL_DPP("a1", "ma", "j1")
            CHOL_DPP("d2", "md", "j2") CHOL_DPP("a2", "ma", "j2")
            : [d0] "+&v"(d[J + 0]), [a0] "+&v"(a[J + 0]), [d1] "+&v"(d[J + 1]), [a1] "+&v"(a[J + 1]), [d2] "+&v"(d[J + 2]), [a2] "+&v"(a[J + 2])
            : [dc] "v"(dc), [md] "v"(md), [ma] "v"(ma), [j0] "n"(J + 0), [j1] "n"(J + 1), [j2] "n"(J + 2));
    } else if constexpr (NJ == 2) {
        asm("s_nop 1\n\t"
            CHOL_DPP("d0", "md", "j0") CHOL_DPP("a0", "ma", "j0")
            CHOL_DPP("d1", "md", "j1") CHOL_DPP("a1", "ma", "j1")
            : [d0] "+&v"(d[J + 0]), [a0] "+&v"(a[J + 0]), [d1] "+&v"(d[J + 1]), [a1] "+&v"(a[J + 1])
            : [dc] "v"(dc), [md] "v"(md), [ma] "v"(ma), [j0] "n"(J + 0), [j1] "n"(J + 1));
    } else if constexpr (NJ == 1) {
        asm("s_nop 1\n\t"
            CHOL_DPP("d0", "md", "j0") CHOL_DPP("a0", "ma", "j0")
            : [d0] "+&v"(d[J + 0]), [a0] "+&v"(a[J + 0])
            : [dc] "v"(dc), [md] "v"(md), [ma] "v"(ma), [j0] "n"(J + 0));
    }
#endif
}
#undef CHOL_DPP
// v of lane J of the lane's row of 16
template <int J>
__device__ __forceinline__ double row_bcast(double v) {
    double x = v;
#if defined(__HIP_DEVICE_COMPILE__)
    asm("s_nop 1\n\tv_mov_b64_dpp %0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf"
        : "=v"(x)
        : "v"(v), "n"(J));
#endif
    return x;
}
// Pivot C: its reciprocal rp is given; that of pivot C + 1 (rcp_newton, in steps) is made
// between the eliminations, five columns at a time.
template <int C>
__device__ __forceinline__ void chol_pivots(double (&d)[16], double (&a)[16], double dg, double piv,
                                            double rp, double &mypiv, bool &inrange, int l16) {
    inrange = inrange && piv >= 0x1p-1000 && piv <= 0x1p+1000;
    mypiv = l16 == C ? piv : mypiv;
    if constexpr (C < 15) {
        constexpr int R = 15 - C, N1 = R < 5 ? R : 5, N2 = R - N1 < 5 ? R - N1 : 5, N3 = R - N1 - N2;
        const double ma = -(a[C] * rp), md = -(d[C] * rp);
        chol_eliminate<C + 1, N1>(d, a, d[C], md, ma);
        const double p1 = row_bcast<C + 1>(dg + d[C + 1]);
        double r1 = __builtin_amdgcn_rcp(p1);
        __builtin_amdgcn_sched_barrier(0);
        chol_eliminate<C + 1 + N1, N2>(d, a, d[C], md, ma);
        r1 = fma(fma(-p1, r1, 1.0), r1, r1);
        __builtin_amdgcn_sched_barrier(0);
        chol_eliminate<C + 1 + N1 + N2, N3>(d, a, d[C], md, ma);
        r1 = fma(fma(-p1, r1, 1.0), r1, r1);
        chol_pivots<C + 1>(d, a, dg, p1, r1, mypiv, inrange, l16);
    }
}
template <int C>
__device__ __forceinline__ void chol_scale(double (&a)[16], double rd, double diag, int own) {
    const double r = row_bcast<C>(rd);
    a[C] = own == C ? diag : a[C] * r;
    if constexpr (C < 15) chol_scale<C + 1>(a, rd, diag, own);
}

// wave 0
__device__ __forceinline__ bool chol_panels(CholLds &T, int lane) {
    double(*S)[CH_LP] = T.S;
    const int l16 = lane & 15;
    bool bad = false;
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        // a: the lane's row; d: row l16 of the diagonal block, in every row of 16 lanes
        double a[16], d[16];
        d2v_t *row = reinterpret_cast<d2v_t *>(&S[lane][16 * p]);
        const d2v_t *drow = reinterpret_cast<const d2v_t *>(&S[16 * p + l16][16 * p]);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const d2v_t u = row[t], x = drow[t];
            a[2 * t] = u.x;
            a[2 * t + 1] = u.y;
            d[2 * t] = x.x;
            d[2 * t + 1] = x.y;
        }
        if (p > 0 && lane < 16)
#pragma unroll
            for (int c = 0; c < 16; ++c) a[c] = lane == c ? 1.0 : 0.0;
        double mypiv = 1.0;
        bool inrange = true;
        // lanes above row j update entries that are never read
        const double dg = T.diag[16 * p + l16], p0 = row_bcast<0>(dg + d[0]);
        chol_pivots<0>(d, a, dg, p0, rcp_newton(p0), mypiv, inrange, l16);
        if (!inrange) {
            // a pivot that is not positive, or outside the range of rcp_newton: the
            // panel again, on its columns in LDS, with divisions
#pragma unroll 1
            for (int c = 0; c < 16; ++c) {
                const int pc = 16 * p + c;
                double piv = T.diag[pc] + S[pc][pc];
                if (!(piv > 0.0) || !isfinite(piv)) {
                    bad = true;
                    piv = 1.0;
                }
                mypiv = l16 == c ? piv : mypiv;
                const double m = S[lane][pc] / piv;
#pragma unroll 1
                for (int j = c + 1; j < 16; ++j)
                    if (lane >= 16 * p + j)
                        S[lane][16 * p + j] = fma(-m, S[16 * p + j][pc], S[lane][16 * p + j]);
            }
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                const d2v_t u = row[t];
                a[2 * t] = u.x;
                a[2 * t + 1] = u.y;
            }
        }
        const double sd = sqrt(mypiv), rd = 1.0 / sd;
        chol_scale<0>(a, rd, sd, lane - 16 * p);
        if (lane >= 16 * p) {
#pragma unroll
            for (int t = 0; t < 8; ++t) row[t] = (d2v_t){a[2 * t], a[2 * t + 1]};
            if (lane < 16 * p + 16) T.rdiag[lane] = rd;
        } else if (lane < 16) {
#pragma unroll
            for (int c = 0; c < 16; ++c) T.Xd[p][c][lane] = a[c];
        }
        if (p > 0 && !inrange) chol_invert16(T, p, lane);
        __syncthreads();
        if (p < 3) __syncthreads();   // column p + 1
    }
    return bad;
}

// waves 1-3: the same barriers
template <class Work>
__device__ __forceinline__ void chol_blocks(CholLds &T, int wave, int lane, Work work) {
    double(*S)[CH_LP] = T.S;
    const int l16 = lane & 15, g4 = lane >> 4;
    // S(i, j) -= L(i, p) L(j, p)^T for 16 x 16 blocks
    auto update = [&](int i, int j, int p) {
        d4_t acc;
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = S[16 * i + g4 + 4 * r][16 * j + l16];
#pragma unroll
        for (int s = 0; s < 4; ++s)
            acc = __builtin_amdgcn_mfma_f64_16x16x4f64(-S[16 * i + l16][16 * p + 4 * s + g4],
                                                       S[16 * j + l16][16 * p + 4 * s + g4], acc, 0,
                                                       0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) S[16 * i + g4 + 4 * r][16 * j + l16] = acc[r];
    };
#pragma unroll
    for (int p = 0; p < 4; ++p) {
        // panel p - 1: the blocks right of column p
        if (p == 1) update(wave == 1 ? 2 : 3, wave == 3 ? 3 : 2, 0);
        if (p == 2 && wave == 1) update(3, 3, 1);
        if (p == 2 && wave == 2) chol_invert16(T, 0, lane);
        work(p);
        __syncthreads();
        if (p < 3) {
            if (wave > p) update(wave, p + 1, p);
            __syncthreads();
        }
    }
}

// Block column `wave` of L11^{-1} on MFMA from the inverses of the diagonal blocks, X(i, j)
// = -X(i, i) sum_k L(i, k) X(k, j); x[k] holds X(k, wave) as l16 = column, g4 + 4 r = row,
// which is also the B operand of step r, so the column stays in registers.
__device__ __forceinline__ void chol_inverse64(const CholLds &T, int wave, int lane, d4_t (&x)[4]) {
    const int l16 = lane & 15, g4 = lane >> 4;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        x[i] = (d4_t){0.0, 0.0, 0.0, 0.0};
        if (i == wave) {
#pragma unroll
            for (int r = 0; r < 4; ++r) x[i][r] = T.Xd[i][g4 + 4 * r][l16];
        } else if (i > wave) {
            d4_t t = (d4_t){0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int k = 0; k < i; ++k)
                if (k >= wave)
#pragma unroll
                    for (int s = 0; s < 4; ++s)
                        t = __builtin_amdgcn_mfma_f64_16x16x4f64(
                            T.S[16 * i + l16][16 * k + 4 * s + g4], x[k][s], t, 0, 0, 0);
#pragma unroll
            for (int s = 0; s < 4; ++s)
                x[i] = __builtin_amdgcn_mfma_f64_16x16x4f64(-T.Xd[i][l16][4 * s + g4], t[s], x[i], 0,
                                                            0, 0);
        }
    }
}

// log-det partial of the block: one log per lane, then a fixed butterfly in double-double
__device__ __forceinline__ void chol_logdet(const CholLds &T, const FragDev &F, int w, int step,
                                            int nbj, int lane) {
    dd_t sl = {lane < nbj ? log(T.S[lane][lane]) : 0.0, 0.0};
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const dd_t o = {__shfl_xor(sl.hi, off), __shfl_xor(sl.lo, off)};
        sl = dd_add(sl, o);
    }
    if (lane == 0) {
        double *part = F.ldpart + ((int64_t)w * F.nsteps + step) * 2;
        part[0] = sl.hi;
        part[1] = sl.lo;
    }
}

// Diagonal block of step `step` of matrix w, one work-group per matrix: linv, log-det
// partial, status, optional L11 write-back.
__global__ __launch_bounds__(256) void k_potrf_diag(const FragDev *__restrict__ fr,
                                                   const int64_t *__restrict__ pre, int nfrag,
                                                   int step) {
    __shared__ __attribute__((aligned(16))) CholLds T;
    __shared__ int64_t s_pre[FIND_LDS_MAX + 1];
    const int64_t b = blockIdx.x;
    const int f = find_frag_lds(pre, nfrag, b, s_pre);
    const int w = (int)(b - (nfrag <= FIND_LDS_MAX ? s_pre[f] : pre[f]));
    const FragDev &F = fr[f];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int N = F.N;
    const int j0 = step * CHOL_NB;
    const int nbj = min(CHOL_NB, N - j0);
    double *A = F.Pi + (int64_t)w * N * N;
    chol_load64(T, (const gdouble_t *)A, N, j0, nbj, wave, lane);
    __syncthreads();
    bool bad = false;
    if (wave == 0)
        bad = chol_panels(T, lane);
    else
        chol_blocks(T, wave, lane, [](int) {});
    if (wave == 3) chol_logdet(T, F, w, step, nbj, lane);
    if (F.keep_l11) {
        // the factored block back into Pi (lower triangle and diagonal); no
        // other work item reads this diagonal block
        for (int r = wave; r < nbj; r += 4)
            if (lane <= r) A[(int64_t)(j0 + r) * N + j0 + lane] = T.S[r][lane];
    }
    d4_t x[4];
    chol_inverse64(T, wave, lane, x);
    double *linv = F.linv + (int64_t)w * CHOL_NB * CHOL_NB;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            linv[(16 * i + (lane >> 4) + 4 * r) * CHOL_NB + 16 * wave + (lane & 15)] = x[i][r];
    if (threadIdx.x == 0 && bad) F.status[w] = 1;
}

// One step of the Cholesky in one launch, for launches of few matrices: work-group (w, r)
// takes the 64 rows from j0 + 64 r of the step's 64 columns.  Every one factors the
// diagonal block itself (wave 0, bound by latency, on CUs that would be idle); meanwhile
// waves 1-3 apply the outer panel's earlier columns to their rows (left-looking, rank 64
// s_in, operands straight from L2).  Then L21 = B L11^{-T}, and the work-groups
// within the outer panel bring their own diagonal block up to date, so that the
// next step finds it complete.
// N = 400, 16 matrices: 22 to 26 us a step of the first outer panel, 13 us the last one;
// E_RPA of o = 8, v = 72 with three launches a step 451 us, with this kernel and k_chol_rest
// 331.
// r = 0 writes the log-det partial and the status.  No work-group may see a half-factored
// block, so with keep_l11 it leaves L11 in linv and copies it into Pi in the next
// step (pend: the previous step did so); the matrix's last step writes it at once.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_chol_step(
    const FragDev *__restrict__ fr, const int64_t *__restrict__ pre, int nfrag, int step, int pend) {
    __shared__ __attribute__((aligned(16))) CholLds T;
    // B, and before it the waves' own stages of 96 rows x 16 columns
    __shared__ __attribute__((aligned(16))) double sm[3 * 96 * 16];
    static_assert(CHOL_NB * CH_LP <= 3 * 96 * 16, "B fits");
    double(*sB)[CH_LP] = reinterpret_cast<double(*)[CH_LP]>(sm);
    const int64_t b = blockIdx.x;
    const int f = __builtin_amdgcn_readfirstlane(find_frag(pre, nfrag, b));
    const FragDev &F = fr[f];
    const int N = F.N;
    const int j0 = step * CHOL_NB;
    const int nrb = (N - j0 + CHOL_NB - 1) / CHOL_NB;
    const int64_t lb = b - pre[f];
    const int w = __builtin_amdgcn_readfirstlane((int)(lb / nrb));
    const int rb = __builtin_amdgcn_readfirstlane((int)(lb - (int64_t)w * nrb));
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int l16 = lane & 15, g4 = lane >> 4;
    const int nbj = min(CHOL_NB, N - j0);
    const int s_in = step % CHOL_OUTER, kbase = j0 - s_in * CHOL_NB;
    double *A = F.Pi + (int64_t)w * N * N;
    const gdouble_t *G = (const gdouble_t *)A;
    gdouble_mut_t *GM = (gdouble_mut_t *)A;
    double *linv = F.linv + (int64_t)w * CHOL_NB * CHOL_NB;
    chol_load64(T, G, N, j0, nbj, wave, lane);
    if (rb == 0) {
        if (pend && F.keep_l11)
            for (int r = wave; r < CHOL_NB; r += 4)
                if (lane <= r) GM[(int64_t)(j0 - CHOL_NB + r) * N + j0 - CHOL_NB + lane] =
                    linv[r * CHOL_NB + lane];
        __syncthreads();
        bool bad = false;
        if (wave == 0)
            bad = chol_panels(T, lane);
        else
            chol_blocks(T, wave, lane, [](int) {});
        if (wave == 3) chol_logdet(T, F, w, step, nbj, lane);
        if (F.keep_l11) {
            const bool last = nrb == 1;
            for (int r = wave; r < nbj; r += 4)
                if (lane <= r) {
                    if (last)
                        GM[(int64_t)(j0 + r) * N + j0 + lane] = T.S[r][lane];
                    else
                        linv[r * CHOL_NB + lane] = T.S[r][lane];
                }
        }
        if (threadIdx.x == 0 && bad) F.status[w] = 1;
        return;
    }
    const int R0 = j0 + CHOL_NB * rb;
    if (wave == 0) {
        __syncthreads();
        chol_panels(T, lane);
    } else {
        // Waves 1-3, v = wave - 1: block row v of B and the blocks (3, v) and, for the last
        // wave, (3, 3); acc = sum P_r P_d^T - A
        const int v = wave - 1;
        d4_t acc[6];
        auto brow = [&](int q) { return q < 4 ? v : 3; };
        auto bcol = [&](int q) { return q < 4 ? q : (q == 4 ? v : 3); };
        const int nq = wave == 3 ? 6 : 5;
#pragma unroll
        for (int q = 0; q < 6; ++q)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = R0 + 16 * brow(q) + g4 + 4 * r;
                acc[q][r] = -G[(int64_t)min(row, N - 1) * N + j0 + 16 * bcol(q) + l16];
            }
        // 16 columns of the outer panel, rows of blocks v and 3 of the work-group and of the
        // diagonal block's four: four rows per load, then through LDS (k pairs swizzled as in
        // gemm_tile.h), the wave's own rows only, so without a barrier.  Straight into the
        // MFMA layout, 16 rows x 32 bytes per load, 4500 cycles per 16 columns instead
        // of 3000.
        double *st = sm + 96 * 16 * v;
        double x[6][4];
        uint32_t roff[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                roff[h][q] = (uint32_t)min((h == 0 ? 16 * v : 48) + 4 * q + g4, N - 1 - R0) * (uint32_t)N + l16;
        auto fetch = [&](int g) {
            const gdouble_t *pr = G + (int64_t)R0 * N + kbase + 16 * g;
            const gdouble_t *pd = G + (int64_t)j0 * N + kbase + 16 * g;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int q = 0; q < 4; ++q) x[h][q] = pr[roff[h][q]];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    x[2 + i][q] = pd[(int64_t)(16 * i + 4 * q) * N + (uint32_t)(g4 * N + l16)];
        };
        if (s_in > 0) fetch(0);
        __syncthreads();
        chol_blocks(T, wave, lane, [&](int p) {
            for (int g = p * s_in; g < (p + 1) * s_in; ++g) {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
                for (int i = 0; i < 6; ++i)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        st[(16 * i + 4 * q + g4) * 16 + 2 * ((l16 >> 1) ^ (2 * q + (g4 >> 1))) + (l16 & 1)] =
                            x[i][q];
                fetch(min(g + 1, 4 * s_in - 1));
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                auto frag = [&](int i, int h) {
                    return *reinterpret_cast<const d2v_t *>(
                        &st[(16 * i + l16) * 16 + 2 * ((2 * g4 + h) ^ (l16 >> 1))]);
                };
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    d2v_t fr[6];
#pragma unroll
                    for (int i = 0; i < 6; ++i) fr[i] = frag(i, h);
                    const d2v_t dv = frag(2 + v, h);
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
#pragma unroll
                        for (int q = 0; q < 4; ++q)
                            acc[q] = __builtin_amdgcn_mfma_f64_16x16x4f64(fr[0][k], fr[2 + q][k], acc[q], 0, 0, 0);
                        acc[4] = __builtin_amdgcn_mfma_f64_16x16x4f64(fr[1][k], dv[k], acc[4], 0, 0, 0);
                        if (nq == 6)
                            acc[5] = __builtin_amdgcn_mfma_f64_16x16x4f64(fr[1][k], fr[5][k], acc[5], 0, 0, 0);
                    }
                }
            }
        });
#pragma unroll
        for (int q = 0; q < 6; ++q)
            if (q < nq)
#pragma unroll
                for (int r = 0; r < 4; ++r) sB[16 * brow(q) + g4 + 4 * r][16 * bcol(q) + l16] = -acc[q][r];
    }
    __syncthreads();
    // Block row `wave` of L21, transposed: X_c = L(c, c)^{-1} (B_c^T - sum_{k<c} L(c, k) X_k),
    // X_k as l16 = row, g4 + 4 r = column, which is also the B operand of step r.
    // 3100 cycles; by way of the whole L11^{-1} 7900.
    d4_t l21[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        d4_t t;
#pragma unroll
        for (int r = 0; r < 4; ++r) t[r] = sB[16 * wave + l16][16 * c + g4 + 4 * r];
#pragma unroll
        for (int k = 0; k < c; ++k)
#pragma unroll
            for (int s = 0; s < 4; ++s)
                t = __builtin_amdgcn_mfma_f64_16x16x4f64(-T.S[16 * c + l16][16 * k + 4 * s + g4],
                                                         l21[k][s], t, 0, 0, 0);
        l21[c] = (d4_t){0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < 4; ++s)
            l21[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(T.Xd[c][l16][4 * s + g4], t[s], l21[c], 0, 0, 0);
    }
    // through the wave's own rows of B to whole rows
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) sB[16 * wave + l16][16 * c + g4 + 4 * r] = l21[c][r];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int row = R0 + 16 * wave + r;
        if (row < N) GM[(int64_t)row * N + j0 + lane] = sB[16 * wave + r][lane];
    }
    if (rb > CHOL_OUTER - 1 - s_in) return;
    // the work-group's own diagonal block -= L21 L21^T (lower blocks)
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (j > wave) break;
        d4_t t = (d4_t){0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < 16; ++s)
            t = __builtin_amdgcn_mfma_f64_16x16x4f64(sB[16 * wave + l16][4 * s + g4],
                                                     sB[16 * j + l16][4 * s + g4], t, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = R0 + 16 * wave + g4 + 4 * r, col = R0 + 16 * j + l16;
            if (row < N && col <= row) GM[(int64_t)row * N + col] -= t[r];
        }
    }
}

// One step's 64 rows from j0 + 64 r of its 64 columns, for launches of many matrices (the
// diagonal block is k_potrf_diag's): B = A - sum P_r P_d^T over the outer panel's earlier
// columns by the loop of k_gemm_f64 (left-looking, rank 64 s_in), L21 = B L11^{-T} with the
// inverse in LDS, and within the outer panel the update of the work-group's own diagonal
// block, so that the next k_potrf_diag finds it complete.  B passes from the product to the
// solve in the product's stage buffers, 16 rows in each: 66 KB of LDS, two
// work-groups per CU.  Bound by the latencies between its short phases: 32 fragments of
// the batch shapes, 20 launches, 3.1 ms (a strip kernel that kept C in memory and a
// triangular solve of its own: 4.0 ms).
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_chol_panel(
    const FragDev *__restrict__ fr, const int64_t *__restrict__ pre, int nfrag, int step) {
    constexpr int T = CHOL_NB;
    static_assert(gemm_lds<true>(T) == 16 * T, "a stage buffer holds 16 rows of B");
    __shared__ __attribute__((aligned(16))) double sA0[gemm_lds<true>(T)], sA1[gemm_lds<true>(T)];
    __shared__ __attribute__((aligned(16))) double sB0[gemm_lds<true>(T)], sB1[gemm_lds<true>(T)];
    __shared__ __attribute__((aligned(16))) double sL[T][CH_LP];
    const int64_t b = blockIdx.x;
    const int f = __builtin_amdgcn_readfirstlane(find_frag(pre, nfrag, b));
    const FragDev &F = fr[f];
    const int N = F.N;
    const int j0 = step * CHOL_NB;
    const int nrb = (N - j0 + CHOL_NB - 1) / CHOL_NB - 1;
    const int64_t lb = b - pre[f];
    const int w = __builtin_amdgcn_readfirstlane((int)(lb / nrb));
    const int rb = 1 + __builtin_amdgcn_readfirstlane((int)(lb - (int64_t)w * nrb));
    const int R0 = j0 + CHOL_NB * rb;
    const int s_in = step % CHOL_OUTER, kbase = j0 - s_in * CHOL_NB;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int l16 = lane & 15, g4 = lane >> 4, wm = wave >> 1, wn = wave & 1;
    double *A = F.Pi + (int64_t)w * N * N;
    gdouble_mut_t *G = (gdouble_mut_t *)A;
    const gdouble_t *linv = (const gdouble_t *)F.linv + (int64_t)w * CHOL_NB * CHOL_NB;
    // B in accumulator layout: row 32 wn + 16 j + g4 + 4 r, column 32 wm + 16 i + l16
    d4_t a[2][2], acc[2][2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = min(R0 + 32 * wn + 16 * j + g4 + 4 * r, N - 1);
                a[i][j][r] = G[(int64_t)row * N + j0 + 32 * wm + 16 * i + l16];
                acc[i][j][r] = 0.0;
            }
#pragma unroll
    for (int r = 0; r < 16; ++r) sL[4 * r + wave][lane] = linv[(4 * r + wave) * CHOL_NB + lane];
    if (s_in > 0)
        gemm_tile<true, true, T>(acc, A, N, j0, N, A, N, R0, N, kbase, j0, j0, true, sA0, sA1, sB0,
                                 sB1);
    __syncthreads();   // the stage buffers are read
    // row q of B's block row c, columns XOR-swizzled by 4 q
    auto rows = [&](int c) { return c < 2 ? (c == 0 ? sA0 : sA1) : (c == 2 ? sB0 : sB1); };
    auto at = [](int q, int col) { return q * CHOL_NB + (col ^ (4 * q)); };
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        double *L = rows(2 * wn + j);
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                L[at(g4 + 4 * r, 32 * wm + 16 * i + l16)] = a[i][j][r] - acc[i][j][r];
    }
    __syncthreads();
    // block row `wave` of L21, transposed: X_c = sum_{k <= c} L11^{-1}(c, k) B_k^T
    double *own = rows(wave);
    d4_t bt[4], x[4];
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) bt[c][r] = own[at(l16, 16 * c + g4 + 4 * r)];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        x[c] = (d4_t){0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int k = 0; k <= c; ++k)
#pragma unroll
            for (int s = 0; s < 4; ++s)
                x[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(sL[16 * c + l16][16 * k + 4 * s + g4],
                                                            bt[k][s], x[c], 0, 0, 0);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int r = 0; r < 4; ++r) own[at(l16, 16 * c + g4 + 4 * r)] = x[c][r];
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int row = R0 + 16 * wave + r;
        if (row < N) G[(int64_t)row * N + j0 + lane] = own[at(r, lane)];
    }
    if (rb > CHOL_OUTER - 1 - s_in) return;
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (j > wave) break;
        const double *oj = rows(j);
        d4_t t = (d4_t){0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int s = 0; s < 16; ++s)
            t = __builtin_amdgcn_mfma_f64_16x16x4f64(own[at(l16, 4 * s + g4)], oj[at(l16, 4 * s + g4)], t,
                                                     0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = R0 + 16 * wave + g4 + 4 * r, col = R0 + 16 * j + l16;
            if (row < N && col <= row) G[(int64_t)row * N + col] -= t[r];
        }
    }
}

constexpr int REST_T = 64;   // tile edge of the rest

// Rank-256 update of the trailing matrix, one 64 x 64 tile (ti >= tj) per work-group:
// C -= P_i P_j^T by the loop of k_gemm_f64 (both panels are rows of A, contiguous in
// k), then one read and write of C's lower part.  Bound by the MFMA pipe where the
// launch is large (2.1 ms at N = 1800, 24 frequencies, 24 fragments) and by the length of
// one tile's loop where it is small.  Four work-groups per CU hide each other's C
// pass, which the 128 x 128 tiles of two per CU did not.  Average launch: N = 400, 16 matrices
// 21 us; N = 1800, 24 matrices 137 us; 24 x 24 of N up to 1800 676 us (128 x 128 tiles:
// 54, 191, 935; register-staged 128 x 128 tiles with C preloaded: 50, 194, 890).
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_chol_rest(
    const FragDev *__restrict__ fr, const int64_t *__restrict__ pre, int nfrag, int step) {
    constexpr int T = REST_T;
    __shared__ __attribute__((aligned(16))) double sA0[gemm_lds<true>(T)], sA1[gemm_lds<true>(T)];
    __shared__ __attribute__((aligned(16))) double sB0[gemm_lds<true>(T)], sB1[gemm_lds<true>(T)];
    const int64_t b = blockIdx.x;
    const int f = __builtin_amdgcn_readfirstlane(find_frag(pre, nfrag, b));
    const FragDev &F = fr[f];
    const int N = F.N;
    const int t0 = (step + 1) * CHOL_NB, kbase = t0 - CHOL_OUTER * CHOL_NB;
    const int nt = (N - t0 + T - 1) / T, nitems = nt * (nt + 1) / 2;
    const int64_t lb = b - pre[f];
    const int w = __builtin_amdgcn_readfirstlane((int)(lb / nitems));
    int ti, tj;
    tri_decode((int)(lb - (int64_t)w * nitems), ti, tj);
    const int Ri = t0 + T * __builtin_amdgcn_readfirstlane(ti);
    const int Rj = t0 + T * __builtin_amdgcn_readfirstlane(tj);
    double *A = F.Pi + (int64_t)w * N * N;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    // the wave's block: columns Rj + T/2 wm .., rows Ri + T/2 wn ..
    const int c0 = Rj + T / 2 * (wave >> 1), r0 = Ri + T / 2 * (wave & 1);
    const bool active = r0 < N && c0 < N && c0 < r0 + T / 2;
    constexpr int NB = T / 32;
    d4_t acc[NB][NB];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) acc[i][j] = (d4_t){0.0, 0.0, 0.0, 0.0};
    gemm_tile<true, true, T>(acc, A, N, Rj, N, A, N, Ri, N, kbase, t0, t0, active, sA0, sA1, sB0,
                             sB1);
    if (!active) return;
    gdouble_mut_t *C = (gdouble_mut_t *)A;
#pragma unroll
    for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = r0 + 16 * j + (lane >> 4) + 4 * r;
#pragma unroll
            for (int i = 0; i < NB; ++i) {
                const int col = c0 + 16 * i + (lane & 15);
                if (row < N && col <= row) C[(int64_t)row * N + col] -= acc[i][j][r];
            }
        }
}

int64_t chol_items(int list, int64_t N, int64_t F, int64_t j) {
    const int64_t j0 = j * CHOL_NB, t0 = j0 + CHOL_NB;
    const bool rest = j % CHOL_OUTER == CHOL_OUTER - 1;
    auto tiles = [&](int64_t t) { return N > t0 ? (N - t0 + t - 1) / t : 0; };
    switch (list) {
    case CHOL_DIAG: return N > j0 ? F : 0;
    case CHOL_PANEL: return F * tiles(CHOL_NB);
    case CHOL_REST: return rest ? F * tiles(REST_T) * (tiles(REST_T) + 1) / 2 : 0;
    default: return N > j0 ? F * (1 + tiles(CHOL_NB)) : 0;   // CHOL_STEP
    }
}

int launch_cholesky(brpa_ctx *ctx, const FragDev *fr, int nfrag, int nsteps, const int64_t *d_pre,
                    const int64_t *h_pre) {
    const int64_t ncu = ctx->ncu > 0 ? ctx->ncu : 256;
    bool fused = false, pend = false;
    for (int j = 0; j < nsteps; ++j) {
        auto at = [&](int list) { return ((int64_t)list * nsteps + j) * (nfrag + 1); };
        auto total = [&](int list) { return h_pre[at(list) + nfrag]; };
        auto launch = [&](auto kernel, int list, auto... extra) -> int {
            if (total(list) <= 0) return BRPA_OK;
            hipLaunchKernelGGL(kernel, dim3(grid1(total(list))), dim3(256), 0, ctx->stream, fr,
                               d_pre + at(list), nfrag, j, extra...);
            LAUNCH_CHECK(ctx);
            return BRPA_OK;
        };
        // From the first outer panel on whose steps have at most four work-groups per CU (two
        // rounds of the resident ones) one launch per step.  ERPA of N = 400 / 16 matrices,
        // N = 1053 / 16 and N = 1800 / 24: 411, 2762 and 7471 us with separate launches throughout,
        // 333, 2524 and 7254 us with a line at two per CU, 333, 2526 and 7163 us at four,
        // no different at eight and sixteen.
        if (j % CHOL_OUTER == 0 && !fused) fused = total(CHOL_STEP) <= 4 * ncu;
        if (fused) {
            BRPA_TRY(launch(k_chol_step, CHOL_STEP, pend ? 1 : 0));
            pend = true;
        } else {
            BRPA_TRY(launch(k_potrf_diag, CHOL_DIAG));
            BRPA_TRY(launch(k_chol_panel, CHOL_PANEL));
        }
        BRPA_TRY(launch(k_chol_rest, CHOL_REST));
    }
    return BRPA_OK;
}

// E(u_w) = 2 sum_j log L_jj - tr Pi_w and the quadrature sum of one fragment per
// work-group, all in double-double.  Each of the 16 waves takes one frequency at a
// time (lanes along the diagonal, fixed butterflies); thread 0 adds the weighted
// terms in frequency order.  Latency-bound: the frequencies one after the other on
// four waves, with a barrier per level of their reduction, took 45 us at F = 16,
// N = 400 and 195 us at F = 24, N = 1800; this form takes 7 and 36 us.
constexpr int EN_WAVES = 16;
__global__ __launch_bounds__(64 * EN_WAVES) void k_energy(const FragDev *__restrict__ fr) {
    const FragDev &F = fr[blockIdx.x];
    __shared__ double sh[EN_WAVES], sl[EN_WAVES];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // only this fragment's own Cholesky steps wrote a partial
    const int ns = (F.N + CHOL_NB - 1) / CHOL_NB;
    dd_t etot = {0.0, 0.0};
    for (int w0 = 0; w0 < F.F; w0 += EN_WAVES) {
        const int w = w0 + wave;
        if (w < F.F) {
            dd_t tr = {0.0, 0.0}, ld = {0.0, 0.0};
            for (int P = lane; P < F.N; P += 64) tr = dd_add(tr, F.diag[(int64_t)w * F.N + P]);
            for (int j = lane; j < ns; j += 64) {
                const double *p = F.ldpart + ((int64_t)w * F.nsteps + j) * 2;
                ld = dd_add(ld, (dd_t){p[0], p[1]});
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                const dd_t a = {__shfl_xor(tr.hi, off), __shfl_xor(tr.lo, off)};
                const dd_t b = {__shfl_xor(ld.hi, off), __shfl_xor(ld.lo, off)};
                tr = dd_add(tr, a);
                ld = dd_add(ld, b);
            }
            const dd_t eu = dd_add((dd_t){2.0 * ld.hi, 2.0 * ld.lo}, (dd_t){-tr.hi, -tr.lo});
            if (lane == 0) {
                F.eu[w] = eu.hi + eu.lo;
                const double c = F.weights[w] / (2.0 * 3.14159265358979323846);
                const double ph = c * eu.hi;
                sh[wave] = ph;
                sl[wave] = fma(c, eu.hi, -ph) + c * eu.lo;
            }
        }
        __syncthreads();
        if (threadIdx.x == 0)
            for (int q = 0; q < min(EN_WAVES, F.F - w0); ++q) {
                etot = dd_add(etot, sh[q]);
                etot.lo += sl[q];
            }
        __syncthreads();
    }
    if (threadIdx.x == 0) F.energy[0] = etot.hi + etot.lo;
}

int launch_energy(brpa_ctx *ctx, const FragDev *fr, int nfrag) {
    if (nfrag <= 0) return BRPA_OK;
    hipLaunchKernelGGL(k_energy, dim3(nfrag), dim3(64 * EN_WAVES), 0, ctx->stream, fr);
    LAUNCH_CHECK(ctx);
    return BRPA_OK;
}

// Fill n ints with a value (used instead of hipMemsetAsync so that the
// sequence stays valid under stream capture).
__global__ void k_fill_int(int *p, int64_t n, int v) {
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = v;
}

int launch_fill_int(brpa_ctx *ctx, int *p, int64_t n, int v) {
    if (n <= 0) return BRPA_OK;
    hipLaunchKernelGGL(k_fill_int, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, ctx->stream,
                       p, n, v);
    LAUNCH_CHECK(ctx);
    return BRPA_OK;
}
