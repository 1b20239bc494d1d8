// THC SOSEX + 2g cumulant terms (rpa_CCD_corrections_1b2g,
// rpa/rpa_CCD_Corrections.f90:79-290): YU = Yga U_mu by rocBLAS dgemm for a
// chunk of amplitude vectors, then the fused k_thc_1b2g contraction, or, with many
// vectors, the products of YU and U with the integrals formed once.
#include <rocblas/rocblas.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "dense.h"

int rocblas_handle_of(brpa_ctx *ctx, void **h);
int thc_1b2g_npairs(int64_t G);
int launch_thc_1b2g(brpa_ctx *, const double *YU, const double *X, const double *Z, int64_t G,
                    int64_t o, int64_t nmu, double *part, double *diag, int64_t mu0, double *S);

int launch_thc_pairs(brpa_ctx *, const double *Y, const double *X, int64_t G, int64_t v, int64_t o,
                     double *P, int64_t ldp);
int launch_thc_xx(brpa_ctx *, const double *X, int64_t G, int64_t o, double *XX, int64_t ldp);
int launch_swap_occ(brpa_ctx *, const double *W, int64_t v, int64_t o, double *D, int64_t ldd);
int64_t thc_s2_blocks(int64_t G);
int launch_thc_s2(brpa_ctx *, const double *YU, const double *X, const double *Q, int64_t ldq,
                  int64_t G, int64_t o, int64_t nmu, double *part, double *diag, int64_t mu0,
                  const double *U, int64_t K, const double *DU, double *S);
int launch_gemm_f64(brpa_ctx *, bool ta, bool tb, int64_t m, int64_t n, int64_t k, double alpha,
                    const double *A, int64_t lda, const double *B, int64_t ldb, double beta,
                    double *C, int64_t ldc, bool upper);

namespace {

// The explicit form needs 2 G^2 K + G K^2 flop for D = (aj|bi), G^2 o (o + 1) for Q and
// 2 K^2 NT2 for D U on the GEMM (60 TFLOP/s), with about 150 us of launches on small
// sizes; the fused kernel 2 G^2 o NT2 at 27 TFLOP/s.  At o = 36, v = 300, G = 4032 the
// line lies near 500 vectors: 2100 of them take 31 ms explicitly, 98 ms fused.
// Two K x K and two G x K matrices have to fit 64 GB.
bool explicit_pays(int64_t G, int64_t o, int64_t v, int64_t nt) {
    const double g = (double)G, K = (double)o * (double)v, n = (double)nt;
    const double ex = (2 * g * g * K + g * K * K + g * g * o * (o + 1) + 2 * K * K * n) / 60e6 + 150;
    const double fu = 2 * g * g * o * n / 27e6 + 20;
    return ex < fu && o * v <= 46340 && o * (o + 1) / 2 <= 65535 &&
           8.0 * (2 * K * K + 2 * g * K) <= 64e9;
}

}  // namespace

extern "C" {

int brpa_thc_1b2g(brpa_ctx *ctx, const double *Zgh, const double *Xgi, const double *Yga,
                  const double *Uaim, const double *Am, int64_t ngrid, int64_t nocc, int64_t nvir,
                  int64_t nvecs_t2, double *ec1b, double *ec2g, double *eig_sosex, double *eig_2g,
                  double *yxu_diag) {
    if (!ctx) return BRPA_ERR_ARG;
    if (!Zgh || !Xgi || !Yga || !Uaim || !Am || !ec1b || !ec2g || ngrid <= 0 || nocc <= 0 ||
        nvir <= 0 || nvecs_t2 < 0)
        return brpa_fail(ctx, BRPA_ERR_ARG, "brpa_thc_1b2g: bad arguments");
    const int64_t G = ngrid, o = nocc, v = nvir, nt = nvecs_t2;
    if (G > 65536 || o * v > INT32_MAX || G * std::max(o, v) > INT32_MAX)
        return brpa_fail(ctx, BRPA_ERR_ARG, "brpa_thc_1b2g: sizes beyond the supported range");
    *ec1b = *ec2g = 0.0;
    if (nt == 0) return BRPA_OK;
    BRPA_HIP(ctx, hipSetDevice(ctx->device));
    void *hv = nullptr;
    BRPA_TRY(rocblas_handle_of(ctx, &hv));
    rocblas_handle h = static_cast<rocblas_handle>(hv);
    std::vector<double> a(nt);
    if (is_device_ptr(Am))
        BRPA_TRY(copy_sync(ctx, a.data(), Am, 8 * nt, hipMemcpyDeviceToHost));
    else
        std::memcpy(a.data(), Am, 8 * nt);
    const int npairs = thc_1b2g_npairs(G);
    bool ex = explicit_pays(G, o, v, nt);
    const int64_t K = o * v;
    // leading dimensions of the explicit form's own matrices: a multiple of 16 bytes, for loads
    // on that boundary (TN 4096^3: 1945 us with an odd one, 1893 with an even one; a
    // padded copy of an operand that the caller gave would cost as much)
    const int64_t gp = G + (G & 1), kp = K + (K & 1), L = o * (o + 1) / 2;
    // amplitude vectors per chunk: YU (G x o per vector) below ~1 GB, at most 65535
    const int64_t nmu = std::max<int64_t>(
        1, std::min<int64_t>({nt, (int64_t)65535, (int64_t)(128ll << 20) / (G * o)}));
    const bool zdev = is_device_ptr(Zgh), xdev = is_device_ptr(Xgi), ydev = is_device_ptr(Yga),
               udev = is_device_ptr(Uaim), ddev = yxu_diag && is_device_ptr(yxu_diag);
    const double *dZ = Zgh, *dX = Xgi, *dY = Yga, *dU = Uaim;
    double *YU, *part, *S, *dD = yxu_diag;
    double *P, *ZP, *Q, *W, *D, *DU, *splitws = nullptr;
    const int64_t nsplit = (int64_t)1 << 24;   // the GEMM's split-k partials: 128 MB
    auto layout = [&](Arena &ar) {
        if (!zdev) dZ = ar.take<double>(G * G);
        if (!xdev) dX = ar.take<double>(G * o);
        if (!ydev) dY = ar.take<double>(G * v);
        if (!udev) dU = ar.take<double>(v * o * nt);
        if (yxu_diag && !ddev) dD = ar.take<double>(G * nt);
        YU = ar.take<double>(G * o * nmu);
        part = ar.take<double>(ex ? thc_s2_blocks(G) * nmu : (int64_t)npairs * nmu * 2);
        S = ar.take<double>(2 * nt);
        if (!ex) return;
        P = ar.take<double>(gp * std::max(K, L));
        ZP = ar.take<double>(gp * K);
        Q = ar.take<double>(gp * L);
        W = ar.take<double>(K * K);
        D = ar.take<double>(kp * K);
        DU = ar.take<double>(K * nt);
        splitws = ar.take<double>(nsplit);
    };
    // the explicit form where its buffers are affordable
    Arena count, ar;
    layout(count);
    if (ex && (!ws_affords(ctx, count.off) ||
               ws_reserve(ctx, count.off, &ar) == BRPA_ERR_OOM)) {
        ex = false;
        count = Arena{};
        layout(count);
    }
    BRPA_TRY(ws_reserve(ctx, count.off, &ar));
    dZ = Zgh;
    dX = Xgi;
    dY = Yga;
    dU = Uaim;
    dD = yxu_diag;
    layout(ar);
    if (!zdev) BRPA_TRY(copy_sync(ctx, const_cast<double *>(dZ), Zgh, 8 * G * G, hipMemcpyHostToDevice));
    if (!xdev) BRPA_TRY(copy_sync(ctx, const_cast<double *>(dX), Xgi, 8 * G * o, hipMemcpyHostToDevice));
    if (!ydev) BRPA_TRY(copy_sync(ctx, const_cast<double *>(dY), Yga, 8 * G * v, hipMemcpyHostToDevice));
    if (!udev)
        BRPA_TRY(copy_sync(ctx, const_cast<double *>(dU), Uaim, 8 * v * o * nt, hipMemcpyHostToDevice));
    BRPA_TRY(rocblas_set_stream(h, ctx->stream) == rocblas_status_success
                 ? BRPA_OK
                 : brpa_fail(ctx, BRPA_ERR_SOLVER, "rocblas_set_stream failed"));
    BRPA_HIP(ctx, hipEventRecord(ctx->ev0, ctx->stream));
    const double one = 1.0, zero = 0.0;
    const KstatDrop kdrop{ctx};
    struct SplitLend {
        brpa_ctx *c;
        ~SplitLend() {
            c->split_ws = nullptr;
            c->split_ws_cap = 0;
        }
    } lend{ctx};
    if (ex) {
        ctx->split_ws = splitws;
        ctx->split_ws_cap = (size_t)nsplit;
        // Q = Z XX, D from P^T (Z P); Z is symmetric, so every product is TN
        BRPA_TRY(launch_thc_xx(ctx, dX, G, o, P, gp));
        BRPA_TRY(launch_gemm_f64(ctx, true, false, G, L, G, 1.0, dZ, G, P, gp, 0.0, Q, gp, false));
        BRPA_TRY(launch_thc_pairs(ctx, dY, dX, G, v, o, P, gp));
        BRPA_TRY(launch_gemm_f64(ctx, true, false, G, K, G, 1.0, dZ, G, P, gp, 0.0, ZP, gp, false));
        BRPA_TRY(launch_gemm_f64(ctx, true, false, K, K, G, 1.0, P, gp, ZP, gp, 0.0, W, K, true));
        BRPA_TRY(launch_swap_occ(ctx, W, v, o, D, kp));
        // D U of every vector in one product (its grid is too small chunk by chunk)
        BRPA_TRY(launch_gemm_f64(ctx, true, false, K, nt, K, 1.0, D, kp, dU, K, 0.0, DU, K, false));
    }
    for (int64_t mu0 = 0; mu0 < nt; mu0 += nmu) {
        const int64_t m = std::min(nmu, nt - mu0);
        // YU(:, i + o mu) = Yga U(:, i, mu): column-major G x (o m), K = v
        if (rocblas_dgemm(h, rocblas_operation_none, rocblas_operation_none, (rocblas_int)G,
                          (rocblas_int)(o * m), (rocblas_int)v, &one, dY, (rocblas_int)G,
                          dU + v * o * mu0, (rocblas_int)v, &zero, YU, (rocblas_int)G) !=
            rocblas_status_success)
            return brpa_fail(ctx, BRPA_ERR_SOLVER, "brpa_thc_1b2g: rocblas_dgemm failed");
        if (ex) {
            BRPA_TRY(launch_thc_s2(ctx, YU, dX, Q, gp, G, o, m, part, yxu_diag ? dD : nullptr, mu0,
                                   dU + K * mu0, K, DU + K * mu0, S));
            continue;
        }
        BRPA_TRY(launch_thc_1b2g(ctx, YU, dX, dZ, G, o, m, part, yxu_diag ? dD : nullptr, mu0, S));
    }
    BRPA_HIP(ctx, hipEventRecord(ctx->ev1, ctx->stream));
    // While the device works: the pages of a host diagonal are touched (their contents stay),
    // so that the copy at the end does not fault them in one by one.  G = 4032, 2100
    // vectors, 68 MB of fresh pages: 35.3 ms without, 32.7.
    if (yxu_diag && !ddev)
        for (size_t b = 0, n = 8 * (size_t)(G * nt); b < n; b += 4096) {
            volatile char *p = reinterpret_cast<char *>(yxu_diag) + b;
            *p = *p;
        }
    std::vector<double> hs(2 * nt);
    BRPA_TRY(copy_sync(ctx, hs.data(), S, 8 * 2 * nt, hipMemcpyDeviceToHost));
    if (yxu_diag && !ddev) BRPA_TRY(copy_sync(ctx, yxu_diag, dD, 8 * G * nt, hipMemcpyDeviceToHost));
    float ms = 0.f;
    BRPA_HIP(ctx, hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
    ctx->last_kernel_ms = ms;
    // Ec2g = 2 sum_mu (-2 S2g A^2), Ec1b = 2 sum_mu (-S1b A) (rpa_CCD_Corrections.f90:137-160)
    long double e2 = 0.0L, e1 = 0.0L;
    for (int64_t mu = 0; mu < nt; ++mu) {
        const double s2 = hs[2 * mu], s1 = hs[2 * mu + 1];
        e2 += -2.0L * s2 * a[mu] * a[mu];
        e1 += -(long double)s1 * a[mu];
        if (eig_2g) eig_2g[mu] = -4.0 * s2 * a[mu] * a[mu];
        if (eig_sosex) eig_sosex[mu] = -s1 * a[mu];
    }
    *ec2g = (double)(2.0L * e2);
    *ec1b = (double)(2.0L * e1);
    return BRPA_OK;
}

}  // extern "C"
