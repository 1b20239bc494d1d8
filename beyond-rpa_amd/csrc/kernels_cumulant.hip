// THC SOSEX + 2g cumulant terms (rpa_CCD_corrections_1b2g,
// rpa/rpa_CCD_Corrections.f90:79-290).  For every amplitude vector mu:
//
//   M_mu(g, h) = sum_i YU_mu(g, i) X(h, i),   YU_mu = Y U_mu  (Y = Yga, X = Xgi)
//   S2g_mu = sum_{g,h} Z(g, h) M_mu(g, h)^2
//   S1b_mu = sum_{g,h} Z(g, h) M_mu(g, h) M_mu(h, g)
//
// with Z = Zgh symmetric.  The reference stores M_mu (NGrid x NGrid) per mu and
// walks it by lower-triangular block pairs; here one work-group takes one block
// pair (p >= q) of 64 x 64 grid points and one mu, builds both M(g-block,
// h-block) and M(h-block, g-block)^T in registers on v_mfma_f64_16x16x4_f64
// (K = NOcc, operands straight from L2), contracts them with the Z tile and
// writes two partial sums; M never reaches memory.  The partials are reduced
// per mu in a fixed order (double-double), so the result does not depend on
// scheduling.
//
// With many vectors it costs less to form what does not depend on mu once
// (thc_1b2g_explicit in cumulant.cpp):
//   S2g_mu = sum_g sum_{ij} YU(g, i) YU(g, j) Q(g, ij),  Q = Z (X_i o X_j),
//   S1b_mu = U_mu^T D U_mu,  D(ai, bj) = (aj|bi) = (P^T Z P)(aj, bi),
//            P(g, aj) = Y(g, a) X(g, j).
// The products run on the library's GEMM; here are the kernels around them:
//   k_thc_pairs, k_thc_xx  P and the X_i o X_j, i >= j
//   k_swap_occ             D from the upper triangle of P^T Z P
//   k_thc_s2               S2g partials and the diagonal M_mu(g, g)
//   k_thc_terms            both sums of each vector
#include <algorithm>

#include "device_common.h"
#include "internal.h"

#define LAUNCH_CHECK(ctx)                                                                      \
    do {                                                                                       \
        hipError_t _e = hipGetLastError();                                                     \
        if (_e != hipSuccess)                                                                  \
            return brpa_fail((ctx), BRPA_ERR_HIP, "kernel launch failed: %s (%s:%d)",          \
                             hipGetErrorString(_e), __FILE__, __LINE__);                       \
    } while (0)

namespace {

constexpr int CB = 64;   // grid points per block

// (p, q) with p >= q from the lower-triangle pair index t = p (p + 1) / 2 + q
__device__ __forceinline__ void pair_decode(int t, int &p, int &q) {
    int pp = (int)((sqrt(8.0 * (double)t + 1.0) - 1.0) * 0.5);
    while ((pp + 1) * (pp + 2) / 2 <= t) ++pp;
    while (pp * (pp + 1) / 2 > t) --pp;
    p = pp;
    q = t - pp * (pp + 1) / 2;
}

// grid: x = block pair, y = mu within the chunk.  YU: column-major G x (o nmu)
// (YU_mu(g, i) at g + G (i + o mu)); X: G x o; Z: G x G symmetric.
// part[(mu * npairs + pair) * 2 + {0, 1}] = (S2g, S1b) of the block pair;
// diag (may be null): M_mu(g, g) at g + G (mu0 + mu).
__global__ __launch_bounds__(256) void k_thc_1b2g(const double *__restrict__ YU,
                                                  const double *__restrict__ X,
                                                  const double *__restrict__ Z, int G, int o,
                                                  int npairs, double *__restrict__ part,
                                                  double *__restrict__ diag, int64_t mu0) {
    __shared__ double red[2][4];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int pair = blockIdx.x, mu = blockIdx.y;
    int pb, qb;
    pair_decode(pair, pb, qb);
    const int g0 = pb * CB, h0 = qb * CB;
    const int wm = wave >> 1, wn = wave & 1;
    const double *yu = YU + (int64_t)G * o * mu;

    d4_t P[2][2], Q[2][2];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            P[i][j] = (d4_t){0.0, 0.0, 0.0, 0.0};
            Q[i][j] = (d4_t){0.0, 0.0, 0.0, 0.0};
        }
    // lane rows: m = l % 16 within each 16-row MFMA block, k = l / 16
    const int lm = lane & 15, lk = lane >> 4;
    for (int k0 = 0; k0 < o; k0 += 4) {
        const int k = k0 + lk;
        const bool kin = k < o;
        double ay[2], ax[2], by[2], bx[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int g = g0 + 32 * wm + 16 * i + lm;
            const bool in = kin && g < G;
            ay[i] = in ? yu[g + (int64_t)G * k] : 0.0;
            ax[i] = in ? X[g + (int64_t)G * k] : 0.0;
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int h = h0 + 32 * wn + 16 * j + lm;
            const bool in = kin && h < G;
            by[j] = in ? yu[h + (int64_t)G * k] : 0.0;
            bx[j] = in ? X[h + (int64_t)G * k] : 0.0;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                // P(g, h) = M(g, h) = sum_k YU(g, k) X(h, k); Q(g, h) = M(h, g)
                P[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ay[i], bx[j], P[i][j], 0, 0, 0);
                Q[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(ax[i], by[j], Q[i][j], 0, 0, 0);
            }
    }
    const bool offd = pb != qb;
    double s2 = 0.0, s1 = 0.0;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int g = g0 + 32 * wm + 16 * i + lk + 4 * r;
                const int h = h0 + 32 * wn + 16 * j + lm;
                if (g < G && h < G) {
                    const double z = Z[h + (int64_t)G * g];   // Z(g, h) = Z(h, g)
                    const double p = P[i][j][r], q = Q[i][j][r];
                    if (offd) {
                        s2 += z * (p * p + q * q);
                        s1 += 2.0 * z * p * q;
                    } else {
                        s2 += z * p * p;
                        s1 += z * p * q;
                        if (diag && g == h) diag[g + (int64_t)G * (mu0 + mu)] = p;
                    }
                }
            }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        s2 += __shfl_xor(s2, off);
        s1 += __shfl_xor(s1, off);
    }
    if (lane == 0) {
        red[0][wave] = s2;
        red[1][wave] = s1;
    }
    __syncthreads();
    if (tid == 0) {
        double* out = part + ((int64_t)mu * npairs + pair) * 2;
        out[0] = (red[0][0] + red[0][1]) + (red[0][2] + red[0][3]);
        out[1] = (red[1][0] + red[1][1]) + (red[1][2] + red[1][3]);
    }
}

// S[(mu0 + mu) * 2 + c] = sum over pairs of part[(mu * npairs + pair) * 2 + c], in
// pair order per thread stripe, then a fixed tree; double-double accumulation
__global__ __launch_bounds__(256) void k_thc_1b2g_reduce(const double *__restrict__ part,
                                                         int npairs, double *__restrict__ S,
                                                         int64_t mu0) {
    __shared__ dd_t sh[2][256];
    const int mu = blockIdx.x, tid = threadIdx.x;
    dd_t a = {0.0, 0.0}, b = {0.0, 0.0};
    for (int t = tid; t < npairs; t += 256) {
        a = dd_add(a, part[((int64_t)mu * npairs + t) * 2]);
        b = dd_add(b, part[((int64_t)mu * npairs + t) * 2 + 1]);
    }
    sh[0][tid] = a;
    sh[1][tid] = b;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if (tid < k) {
            sh[0][tid] = dd_add(sh[0][tid], sh[0][tid + k]);
            sh[1][tid] = dd_add(sh[1][tid], sh[1][tid + k]);
        }
        __syncthreads();
    }
    if (tid == 0) {
        S[(mu0 + mu) * 2] = sh[0][0].hi + sh[0][0].lo;
        S[(mu0 + mu) * 2 + 1] = sh[1][0].hi + sh[1][0].lo;
    }
}

// P(g, a + v j) = Y(g, a) X(g, j) for the ncol columns a + v j, leading dimension ldp.  The
// grid covers the columns (x) and groups of 256 points (y) within a launch's limits and
// walks on from there.
constexpr int64_t PAIRS_X = 1 << 22, PAIRS_Y = 65535;   // below 2^32 threads, 2^16 groups
__global__ __launch_bounds__(256) void k_thc_pairs(const double *__restrict__ Y,
                                                   const double *__restrict__ X, int64_t G, int v,
                                                   int64_t ncol, double *__restrict__ P, int64_t ldp) {
    for (int64_t c = blockIdx.x; c < ncol; c += gridDim.x) {
        const int j = (int)c / v, a = (int)c - j * v;
        const double *__restrict__ y = Y + G * a, *__restrict__ x = X + G * j;
        for (int64_t g = blockIdx.y * 256 + threadIdx.x; g < G; g += 256 * (int64_t)gridDim.y)
            P[g + ldp * c] = y[g] * x[g];
    }
}

// XX(g, i (i + 1) / 2 + j) = X(g, i) X(g, j), i >= j
__global__ __launch_bounds__(256) void k_thc_xx(const double *__restrict__ X, int G,
                                                double *__restrict__ XX, int64_t ldp) {
    const int g = blockIdx.x * 256 + threadIdx.x;
    int i, j;
    pair_decode(blockIdx.y, i, j);
    if (g < G) XX[g + ldp * blockIdx.y] = X[g + (int64_t)G * i] * X[g + (int64_t)G * j];
}

// D(a + v i, b + v j) = W(a + v j, b + v i) for the symmetric W (K x K, upper triangle
// valid): one 32 x 32 tile of the v x v block of one pair i >= j per work-group.
// W is read along its columns; the block (i, j) of D is written the same way, its
// mirror (j, i) through LDS.  Bound by memory: W's triangle read and D written.
__global__ __launch_bounds__(256) void k_swap_occ(const double *__restrict__ W, int64_t K, int v,
                                                  int nt, double *__restrict__ D, int64_t ldd) {
    __shared__ double t[32][33];
    const int64_t b = blockIdx.x;
    const int pair = (int)(b / (nt * nt)), tile = (int)(b - (int64_t)pair * nt * nt);
    int i, j;
    pair_decode(pair, i, j);
    const int a0 = 32 * (tile % nt), b0 = 32 * (tile / nt);
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int y = ty; y < 32; y += 8) {
        const int a = a0 + tx, bb = b0 + y;
        if (a < v && bb < v) {
            const int64_t r = a + (int64_t)v * j, c = bb + (int64_t)v * i;
            const double x = W[min(r, c) + K * max(r, c)];
            t[y][tx] = x;
            D[a + (int64_t)v * i + ldd * (bb + (int64_t)v * j)] = x;
        }
    }
    if (i == j) return;
    __syncthreads();
    for (int y = ty; y < 32; y += 8) {
        const int a = a0 + y, bb = b0 + tx;
        if (a < v && bb < v) D[bb + (int64_t)v * j + ldd * (a + (int64_t)v * i)] = t[tx][y];
    }
}

// S2g partials: part[mu * ngb + gb] = sum over 64 grid points of sum_{i >= j} (2 -
// delta_ij) Q(g, ij) YU(g, i) YU(g, j), for 8 vectors per wave (grid: x = 64
// points, y = 32 vectors).  A lane holds one point; rows of Q in blocks of four
// keep 32 accumulators per lane, so a column j costs 12 loads for 32 fma.  diag
// (may be null): M_mu(g, g) = sum_i YU(g, i) X(g, i).  Bound by L2 reads of YU
// (o / 8 passes) and Q: 3.5 ms for 2100 vectors at o = 36, G = 4032 (5.9 ms
// without the second column in flight).
constexpr int S2V = 8;
__global__ __launch_bounds__(256) void k_thc_s2(const double *__restrict__ YU,
                                                const double *__restrict__ X,
                                                const double *__restrict__ Q, int64_t ldq, int G,
                                                int o, int nmu, double *__restrict__ part,
                                                double *__restrict__ diag, int64_t mu0) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int gb = blockIdx.x, m0 = blockIdx.y * (4 * S2V) + wave * S2V;
    if (m0 >= nmu) return;
    const int g = gb * 64 + lane;
    const bool ok = g < G;
    const int gc = ok ? g : G - 1;
    const double *yu[S2V];
#pragma unroll
    for (int u = 0; u < S2V; ++u) yu[u] = YU + (int64_t)G * o * min(m0 + u, nmu - 1) + gc;
    const double *__restrict__ Qg = Q + gc;
    double s[S2V];
#pragma unroll
    for (int u = 0; u < S2V; ++u) s[u] = 0.0;
    for (int i0 = 0; i0 < o; i0 += 4) {
        double t[4][S2V];
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int u = 0; u < S2V; ++u) t[q][u] = 0.0;
#pragma unroll 2
        for (int j = 0; j < min(o, i0 + 4); ++j) {
            double qv[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int i = i0 + q;
                const bool in = i < o && j <= i;
                const double x = Qg[ldq * (in ? (int64_t)i * (i + 1) / 2 + j : 0)];
                qv[q] = in ? (j == i ? x : 2.0 * x) : 0.0;
            }
#pragma unroll
            for (int u = 0; u < S2V; ++u) {
                const double y = yu[u][(int64_t)G * j];
#pragma unroll
                for (int q = 0; q < 4; ++q) t[q][u] = fma(qv[q], y, t[q][u]);
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (i0 + q < o)
#pragma unroll
                for (int u = 0; u < S2V; ++u)
                    s[u] = fma(t[q][u], yu[u][(int64_t)G * (i0 + q)], s[u]);
    }
#pragma unroll
    for (int u = 0; u < S2V; ++u) {
        double x = ok ? s[u] : 0.0;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off);
        if (lane == 0 && m0 + u < nmu) part[(int64_t)(m0 + u) * gridDim.x + gb] = x;
    }
    if (!diag || !ok) return;
#pragma unroll
    for (int u = 0; u < S2V; ++u) s[u] = 0.0;
    for (int i = 0; i < o; ++i) {
        const double x = X[g + (int64_t)G * i];
#pragma unroll
        for (int u = 0; u < S2V; ++u) s[u] = fma(yu[u][(int64_t)G * i], x, s[u]);
    }
#pragma unroll
    for (int u = 0; u < S2V; ++u)
        if (m0 + u < nmu) diag[g + (int64_t)G * (mu0 + m0 + u)] = s[u];
}

// S[2 (mu0 + mu)] = sum of the S2g partials, S[2 (mu0 + mu) + 1] = U_mu^T (D U_mu),
// both in double-double: thread stripes in order, then a fixed tree
__global__ __launch_bounds__(256) void k_thc_terms(const double *__restrict__ part, int ngb,
                                                   const double *__restrict__ U, int64_t K,
                                                   const double *__restrict__ DU,
                                                   double *__restrict__ S, int64_t mu0) {
    __shared__ dd_t sh[2][256];
    const int64_t mu = blockIdx.x;
    const int tid = threadIdx.x;
    dd_t a = {0.0, 0.0}, b = {0.0, 0.0};
    for (int t = tid; t < ngb; t += 256) a = dd_add(a, part[mu * ngb + t]);
    for (int64_t k = tid; k < K; k += 256) {
        const double x = U[k + K * mu], y = DU[k + K * mu], p = x * y;
        b = dd_add(b, (dd_t){p, fma(x, y, -p)});
    }
    sh[0][tid] = a;
    sh[1][tid] = b;
    __syncthreads();
    for (int k = 128; k > 0; k >>= 1) {
        if (tid < k) {
            sh[0][tid] = dd_add(sh[0][tid], sh[0][tid + k]);
            sh[1][tid] = dd_add(sh[1][tid], sh[1][tid + k]);
        }
        __syncthreads();
    }
    if (tid == 0) {
        S[(mu0 + mu) * 2] = sh[0][0].hi + sh[0][0].lo;
        S[(mu0 + mu) * 2 + 1] = sh[1][0].hi + sh[1][0].lo;
    }
}

}  // namespace

int launch_thc_pairs(brpa_ctx *ctx, const double *Y, const double *X, int64_t G, int64_t v,
                     int64_t o, double *P, int64_t ldp) {
    const dim3 grid((unsigned)std::min(v * o, PAIRS_X), (unsigned)std::min((G + 255) / 256, PAIRS_Y));
    hipLaunchKernelGGL(k_thc_pairs, grid, dim3(256), 0, ctx->stream, Y, X, G, (int)v, v * o, P, ldp);
    LAUNCH_CHECK(ctx);
    return BRPA_OK;
}

int launch_thc_xx(brpa_ctx *ctx, const double *X, int64_t G, int64_t o, double *XX, int64_t ldp) {
    hipLaunchKernelGGL(k_thc_xx, dim3((unsigned)((G + 255) / 256), (unsigned)(o * (o + 1) / 2)),
                       dim3(256), 0, ctx->stream, X, (int)G, XX, ldp);
    LAUNCH_CHECK(ctx);
    return BRPA_OK;
}

int launch_swap_occ(brpa_ctx *ctx, const double *W, int64_t v, int64_t o, double *D, int64_t ldd) {
    const int64_t nt = (v + 31) / 32, blocks = nt * nt * (o * (o + 1) / 2);
    if (blocks > INT32_MAX)
        return brpa_fail(ctx, BRPA_ERR_ARG, "THC 1b2g: sizes beyond the supported grid");
    hipLaunchKernelGGL(k_swap_occ, dim3((unsigned)blocks), dim3(256), 0, ctx->stream, W, v * o,
                       (int)v, (int)nt, D, ldd);
    LAUNCH_CHECK(ctx);
    return BRPA_OK;
}

int64_t thc_s2_blocks(int64_t G) { return (G + 63) / 64; }

// part: nmu * thc_s2_blocks(G) doubles
int launch_thc_s2(brpa_ctx *ctx, const double *YU, const double *X, const double *Q, int64_t ldq,
                  int64_t G, int64_t o, int64_t nmu, double *part, double *diag, int64_t mu0,
                  const double *U, int64_t K, const double *DU, double *S) {
    const unsigned ngb = (unsigned)thc_s2_blocks(G);
    hipLaunchKernelGGL(k_thc_s2, dim3(ngb, (unsigned)((nmu + 4 * S2V - 1) / (4 * S2V))), dim3(256),
                       0, ctx->stream, YU, X, Q, ldq, (int)G, (int)o, (int)nmu, part, diag, mu0);
    LAUNCH_CHECK(ctx);
    hipLaunchKernelGGL(k_thc_terms, dim3((unsigned)nmu), dim3(256), 0, ctx->stream, part, (int)ngb,
                       U, K, DU, S, mu0);
    LAUNCH_CHECK(ctx);
    return BRPA_OK;
}

int thc_1b2g_npairs(int64_t G) {
    const int64_t nb = (G + CB - 1) / CB;
    return (int)(nb * (nb + 1) / 2);
}

int launch_thc_1b2g(brpa_ctx *ctx, const double *YU, const double *X, const double *Z, int64_t G,
                    int64_t o, int64_t nmu, double *part, double *diag, int64_t mu0, double *S) {
    if (nmu <= 0 || G <= 0) return BRPA_OK;
    const int npairs = thc_1b2g_npairs(G);
    if (nmu > 65535 || G > 65536)
        return brpa_fail(ctx, BRPA_ERR_ARG, "THC 1b2g: sizes beyond the supported grid");
    hipLaunchKernelGGL(k_thc_1b2g, dim3((unsigned)npairs, (unsigned)nmu), dim3(256), 0, ctx->stream,
                       YU, X, Z, (int)G, (int)o, npairs, part, diag, mu0);
    LAUNCH_CHECK(ctx);
    hipLaunchKernelGGL(k_thc_1b2g_reduce, dim3((unsigned)nmu), dim3(256), 0, ctx->stream, part,
                       npairs, S, mu0);
    LAUNCH_CHECK(ctx);
    return BRPA_OK;
}
