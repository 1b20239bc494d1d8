// Split-BF16 Pi(u) build on gfx950 bf16 MFMA (v_mfma_f32_16x16x32_bf16).
//
// X_w = diag(sqrt(c_w)) R is cut into 128-row blocks.  In block b, column P
// gets a power-of-two scale s = 2^(e-8) with max_k |X[k][P]| < 2^e, and every
// element is written as s (n0 + n1 2^-8 + n2 2^-16 + n3 2^-24) with integers
// |n0| <= 256, |n1|,|n2|,|n3| <= 128.  Slice k is stored as the bf16 value
// n_k 2^(-8k), which is exact.  Pi_w[p][q] = sum_b s_p s_q sum_k x_p x_q, and
// the ten slice products of level a+b <= 3 go to three FP32 accumulators:
//   L0  = n0 n0                          (integer sums < 2^24: exact)
//   L1  = (n0 n1 + n1 n0) 2^-8           (integer sums < 2^24 times 2^-8: exact)
//   L23 = levels 2 and 3                 (rounding ~2^-40 relative to Pi)
// Each 128-row block is flushed to FP64 as s_p s_q (L0 + L1 + L23).  The
// dropped level >= 4 products are ~2^-32 relative.  The diagonal (and so
// tr Pi) is then replaced by its exact FP64 value (k_split partials, summed in
// k_set_diag), which removes the systematic diagonal bias of the truncation.
#include "device_common.h"
#include "internal.h"

#define LAUNCH_CHECK(ctx)                                                                      \
    do {                                                                                       \
        hipError_t _e = hipGetLastError();                                                     \
        if (_e != hipSuccess)                                                                  \
            return brpa_fail((ctx), BRPA_ERR_HIP, "kernel launch failed: %s (%s:%d)",          \
                             hipGetErrorString(_e), __FILE__, __LINE__);                       \
    } while (0)

// Work-groups per fragment: nblk * ceil(N/64).  One work-group splits a 128-row x
// 64-column block of R for every frequency in turn (R is read once).  Thread -> column
// tid/4, rows 32 (tid%4) .. +32, in registers; the four threads of a column combine its
// maximum and its diagonal partial by shuffles, and each thread's 32 rows are one
// 64-byte piece of the slices' layout [w][slice][k / 32][column][32].
//
// Bound by the writes of the slices (8 bytes per element and frequency) and about 32 FP64
// operations per element and frequency: 292 us at K = 4853, N = 1053, 16 frequencies
// (495 us with the block in LDS, read three times per frequency).
constexpr int SPF = 8;                    // frequencies per table load
constexpr int SPQ = SPLIT_KB / 4 + 2;     // pitch of a quarter's rows: four threads, four banks

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 4))) void k_split(const FragDev *__restrict__ fr,
                                              const int64_t *__restrict__ pre, int nfrag) {
    // c_w and sqrt(c_w) of the rows
    __shared__ __attribute__((aligned(16))) double sC[SPF][4 * SPQ], sS[SPF][4 * SPQ];
    const int64_t b = blockIdx.x;
    const int f = __builtin_amdgcn_readfirstlane(find_frag(pre, nfrag, b));
    const FragDev &F = fr[f];
    const int N = F.N, K = F.K;
    const int ncc = (N + 63) / 64;
    const int lb = __builtin_amdgcn_readfirstlane((int)(b - pre[f]));
    const int blk = lb / ncc, cc = lb - blk * ncc;
    const int k0 = blk * SPLIT_KB;
    const int tid = threadIdx.x, g = tid & 3;
    const int P = cc * 64 + (tid >> 2);
    const bool colok = P < N;
    typedef __attribute__((address_space(1))) const double gdbl_t;
    const gdbl_t *R = (const gdbl_t *)F.R, *D = (const gdbl_t *)F.dtab;
    double x[32];
#pragma unroll
    for (int j = 0; j < 32; ++j) {
        const int k = k0 + 32 * g + j;
        const bool ok = colok && k < K;
        x[j] = R[ok ? (int64_t)k * N + P : 0];
        x[j] = ok ? x[j] : 0.0;
    }
    for (int w0 = 0; w0 < F.F; w0 += SPF) {
        const int nw = min(SPF, F.F - w0);
        __syncthreads();
        for (int e = tid; e < SPF * SPLIT_KB; e += 256) {
            const int i = e / SPLIT_KB, r = e - i * SPLIT_KB;
            const bool ok = i < nw && k0 + r < K;
            double c = D[ok ? (int64_t)(w0 + i) * K + k0 + r : 0];
            c = ok ? c : 0.0;
            sC[i][r / 32 * SPQ + r % 32] = c;
            sS[i][r / 32 * SPQ + r % 32] = sqrt(c);
        }
        __syncthreads();
        for (int i = 0; i < nw; ++i) {
            const int w = w0 + i;
            const double *cw = &sC[i][g * SPQ], *sw = &sS[i][g * SPQ];
            // the column's maximum, and its exact diagonal partial sum_k c_w(k) R[k][P]^2 in
            // double-double
            double m = 0.0;
            dd_t ds = {0.0, 0.0};
#pragma unroll
            for (int j = 0; j < 32; ++j) {
                asm("" : "+v"(x[j]));   // its square is cheaper made again than kept
                m = fmax(m, fabs(sw[j] * x[j]));
                const double r2 = x[j] * x[j], r2e = fma(x[j], x[j], -r2);
                const double p = cw[j] * r2, pe = fma(cw[j], r2, -p) + cw[j] * r2e;
                ds = dd_add(ds, p);
                ds.lo += pe;
            }
#pragma unroll
            for (int o = 1; o < 4; o *= 2) {
                m = fmax(m, __shfl_xor(m, o));
                ds = dd_add(ds, (dd_t){__shfl_xor(ds.hi, o), __shfl_xor(ds.lo, o)});
            }
            int e = 0;
            if (m > 0.0) frexp(m, &e);   // m = f 2^e, 0.5 <= f < 1  ->  m < 2^e
            if (!colok) continue;
            if (g == 0) {
                const int64_t o = ((int64_t)w * F.nblk + blk) * N + P;
                F.dpart[2 * o] = ds.hi;
                F.dpart[2 * o + 1] = ds.lo;
                F.scale[o] = (m > 0.0) ? ldexpf(1.0f, e - 8) : 0.0f;
            }
            uint16_t *dst = F.sl + (int64_t)w * NSLICE * N * F.Kpad +
                            ((int64_t)(k0 / 32 + g) * N + P) * 32;
#pragma unroll
            for (int r = 0; r < 32; r += 8) {
                uint32_t pk[NSLICE][4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    float v[NSLICE][2];
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        const int j = r + 2 * q + u;
                        double t = ldexp(sw[j] * x[j], 8 - e);   // |t| < 256, exact
                        const double n = rint(t);
                        v[0][u] = (float)n;
                        t -= n;
                        // rounding to multiples of 2^-8 k by adding 1.5 2^(52-8k): exact steps
#pragma unroll
                        for (int sl = 1; sl < NSLICE; ++sl) {
                            const double M = 1.5 * (double)(1ull << (52 - 8 * sl));
                            const double nk = (t + M) - M;
                            v[sl][u] = (float)nk;
                            t -= nk;
                        }
                    }
                    // n 2^-8k is exact in bf16: the float's low 16 bits are zero
#pragma unroll
                    for (int sl = 0; sl < NSLICE; ++sl)
                        pk[sl][q] = __builtin_amdgcn_perm(__float_as_uint(v[sl][1]),
                                                          __float_as_uint(v[sl][0]), 0x07060302u);
                }
#pragma unroll
                for (int sl = 0; sl < NSLICE; ++sl)
                    *reinterpret_cast<uint4 *>(dst + (int64_t)sl * N * F.Kpad + r) =
                        make_uint4(pk[sl][0], pk[sl][1], pk[sl][2], pk[sl][3]);
            }
        }
    }
}

int launch_split(brpa_ctx *ctx, const FragDev *fr, const int64_t *pre, int nfrag, int64_t total) {
    if (total <= 0) return BRPA_OK;
    hipLaunchKernelGGL(k_split, dim3((unsigned)total), dim3(256), 0, ctx->stream, fr, pre, nfrag);
    LAUNCH_CHECK(ctx);
    return BRPA_OK;
}

// ---------------------------------------------------------------------------
// 128x128 tile pair (p-tile >= q-tile) per work-group, 8 waves as 2 (rows) x 4 (cols)
// sub-tiles of 64x32 (2 waves per SIMD).  Only the lower triangle of Pi is written.
// MFMA v_mfma_f32_16x16x32_bf16 operand layout (lane l):
//   A[m = l%16][k = 8*(l/16) .. +7], B[k = 8*(l/16) .. +7][n = l%16],
//   D: 4 floats, D[r] = C[m = 4*(l/16) + r][n = l%16].
// Both operands are columns of X (k contiguous per column), so A and B are
// read from LDS the same way.
//
// Stages of 32 rows go straight from HBM to LDS (global_load_lds_dwordx4, 16 bytes per
// lane, no register staging), double-buffered.  One wave load fills 1 KB = 16 columns x
// 64 bytes (contiguous in memory); lane l lands in column l/4, slot l%4, and fetches
// k-piece (l%4) ^ ((l/16)%4) of that column, so that the MFMA operand reads (16 columns at
// one k-piece per 16 lanes) hit 16 distinct 4-bank groups.
//
// A stage is four blocks of 16 rows, 20 MFMAs each: the block's four slices against the q
// slices of level <= 3.  A slice's fragment is replaced by the next block's as soon as
// its products are issued, so that 160 accumulator registers (three levels in FP32 and the
// FP64 sum) leave room.  The barrier stands before the fourth block, when the wave has
// read everything of the stage: the loads of the stage after the next go into its buffer,
// and the fourth block reads the next stage's operands.  The FP64 sums of a block of
// rows are made under the MFMAs of the next one.  A wave above the diagonal of a
// diagonal tile only stages.
//
// 913 us at K = 4853, N = 1053, 16 frequencies (1408 us with the operands read behind the
// barrier and every wave waiting for its loads there): 1250 TFLOP/s of the 2000 to 2300
// that MFMAs alone reach on random data, counting whole tiles.  Their area is 1.33 times
// N (N + 1) / 2 there (waves past N multiply like the others): 940 TFLOP/s on the triangle.
constexpr int T16 = 128;
constexpr int KS = 32;          // rows per stage (one MFMA k-depth)

typedef __attribute__((address_space(3))) void lds_void_t;

__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void k_syrk_bf16(
    const FragDev *__restrict__ fr, const int64_t *__restrict__ pre, int nfrag) {
    static_assert(SPLIT_KB == 4 * KS, "four stages per scaled block");
    // [side][slice][column][slot] of 16-byte pieces.  Two arrays and not one with an
    // index: the compiler then knows that a read of one does not wait for the loads into the
    // other.
    __shared__ __attribute__((aligned(16))) uint4 sb0[2][NSLICE][T16][4], sb1[2][NSLICE][T16][4];
    __shared__ __attribute__((aligned(16))) float sSc[2 * T16];
    const int64_t b = xcd_chunks(blockIdx.x, gridDim.x);
    const int f = __builtin_amdgcn_readfirstlane(find_frag(pre, nfrag, b));
    const FragDev &F = fr[f];
    const int N = F.N;
    const int nt = (N + T16 - 1) / T16;
    const int npairs = nt * (nt + 1) / 2;
    const int64_t lb = b - pre[f];
    const int w = __builtin_amdgcn_readfirstlane((int)(lb / npairs));
    const int pair = (int)(lb - (int64_t)w * npairs);
    int tp, tq;
    tri_decode(pair, tp, tq);
    const int p0 = __builtin_amdgcn_readfirstlane(tp * T16), q0 = __builtin_amdgcn_readfirstlane(tq * T16);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int wi = wave >> 2, wj = wave & 3;     // 64-row half, 32-col quarter
    const int64_t Kpad = F.Kpad;
    const int nblk = F.nblk, nst = 4 * nblk;

    // A wave loads one slice of one side: 8 groups of 16 columns, and waves 0-3 the
    // scales of 64 columns.  Columns past N are whatever follows (the allocation ends with
    // SL_PAD spare bytes) or repeat column N - 1: they only feed outputs that are never
    // written.
    const int side = wave >> 2, slice = wave & 3;
    const int lpiece = (lane & 3) ^ ((lane >> 4) & 3);
    const uint32_t goff = (uint32_t)((side ? q0 : p0) + (lane >> 2)) * (2 * KS) + 16u * lpiece;
    const char *base = (const char *)(F.sl + ((int64_t)w * NSLICE + slice) * N * Kpad);
    typedef __attribute__((address_space(1))) const float gfloat_t;
    const gfloat_t *scb = (const gfloat_t *)F.scale + (int64_t)w * nblk * N;
    auto issue = [&](int buf, int st) {
#if defined(__HIP_DEVICE_COMPILE__)
        typedef __attribute__((address_space(1))) const char gchar_t;
        // the load's constant offset counts for both addresses: four groups per base
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const char *src = base + ((int64_t)st * 2 * KS * N + 64 * 2 * KS * h);
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
    // The scales of a block of 128 rows: loaded in its first stage, stored in its second, read in
    // its fourth.  The lane's number is made anew each time, which is cheaper than to
    // keep addresses in registers.
    auto lane_again = [] {
        int z = 0;
        asm volatile("" : "+s"(z));
        return (int)__builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, z));
    };
    float sv = 0.f;
    auto scale_load = [&](int blk) {
        const int c = min((wave & 2 ? q0 : p0) + 64 * (wave & 1) + lane_again(), N - 1);
        sv = scb[(int64_t)blk * N + c];
    };
    auto scale_store = [&] {
        if (wave < 4) sSc[64 * wave + lane_again()] = sv;
    };
    issue(0, 0);
    if (tp == tq && 32 * wj > 64 * wi + 63) {
        __syncthreads();
        issue(1, 1);
        for (int st = 0; st < nst; ++st) {
            __syncthreads();
            if ((st & 3) == 1) scale_store();
            if ((st & 3) == 0) scale_load(st >> 2);
            issue(st & 1, min(st + 2, nst - 1));
        }
        __builtin_amdgcn_s_waitcnt(0);
        return;
    }
    const int fo = (lane & 15) * 4 + ((lane >> 4) ^ ((lane >> 2) & 3));
    auto fragp = [&](int buf, int s, int i) {
        return __builtin_bit_cast(bf8_t, (buf ? &sb1[0][s][64 * wi + 16 * i][0] : &sb0[0][s][64 * wi + 16 * i][0])[fo]);
    };
    auto fragq = [&](int buf, int s, int j) {
        return __builtin_bit_cast(bf8_t, (buf ? &sb1[1][s][32 * wj + 16 * j][0] : &sb0[1][s][32 * wj + 16 * j][0])[fo]);
    };
    f4_t L0[4][2], L1[4][2], L23[4][2];
    double acc[4][2][4];
    bf8_t a[NSLICE], bq[NSLICE][2];
    const f4_t zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            L0[i][j] = L1[i][j] = L23[i][j] = zero;
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.0;
        }
    // rows 16 i .. of the block of 128 that ended: its level sums to FP64
    auto flush = [&](int i) {
        const int l = lane_again();
        const f4_t sp = *reinterpret_cast<const f4_t *>(&sSc[64 * wi + 16 * i + 4 * (l >> 4)]);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const float sq = sSc[T16 + 32 * wj + 16 * j + (l & 15)];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const double v = (double)L0[i][j][r] + (double)L1[i][j][r] + (double)L23[i][j][r];
                acc[i][j][r] = fma(v, (double)sp[r] * (double)sq, acc[i][j][r]);
            }
        }
    };
    auto mma = [](const bf8_t &x, const bf8_t &y, const f4_t &c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(x, y, c, 0, 0, 0);
    };
    __syncthreads();
    issue(1, 1);
#pragma unroll
    for (int s = 3; s >= 0; --s) {
        a[s] = fragp(0, s, 0);
#pragma unroll
        for (int j = 0; j < 2; ++j) bq[s][j] = fragq(0, s, j);
    }
    // the last stages load and read stage nst - 1 again, unused
    for (int blk = 0; blk < nblk; ++blk) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const int st = 4 * blk + ks, buf = ks & 1;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int nb = i == 3 ? buf ^ 1 : buf, ni = (i + 1) & 3;
                if (i == 3) {
                    __syncthreads();
                    if (ks == 1) scale_store();
                    if (ks == 0) scale_load(blk);
                    issue(buf, min(st + 2, nst - 1));
                }
                auto both = [&](const bf8_t &x, int s, f4_t (&c)[2]) {
#pragma unroll
                    for (int j = 0; j < 2; ++j) c[j] = mma(x, bq[s][j], c[j]);
                };
                auto next_q = [&](int s) {
                    if (i == 3)
#pragma unroll
                        for (int j = 0; j < 2; ++j) bq[s][j] = fragq(nb, s, j);
                };
                if (ks == 0)
#pragma unroll
                    for (int j = 0; j < 2; ++j) L0[i][j] = L1[i][j] = L23[i][j] = zero;
                if (ks == 3 && i > 0) flush(i - 1);
                both(a[0], 3, L23[i]);
                next_q(3);
                both(a[0], 1, L1[i]);
                both(a[0], 2, L23[i]);
                both(a[0], 0, L0[i]);
                a[0] = fragp(nb, 0, ni);
                both(a[1], 2, L23[i]);
                next_q(2);
                both(a[1], 0, L1[i]);
                both(a[1], 1, L23[i]);
                a[1] = fragp(nb, 1, ni);
                both(a[2], 1, L23[i]);
                next_q(1);
                both(a[2], 0, L23[i]);
                a[2] = fragp(nb, 2, ni);
                both(a[3], 0, L23[i]);
                next_q(0);
                a[3] = fragp(nb, 3, ni);
                if (i < 3 && (ks < 3 || i == 0)) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 8, 0);     // MFMA
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // LDS read
                    __builtin_amdgcn_sched_group_barrier(0x8, 6, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x8, 4, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x8, 2, 0);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                }
                if (ks == 3 && i > 0 && i < 3) {
                    __builtin_amdgcn_sched_group_barrier(0x100, 3, 2);   // scales
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        __builtin_amdgcn_sched_group_barrier(0x8, 1, 2);
                        __builtin_amdgcn_sched_group_barrier(0x2, 5, 2);     // VALU
                    }
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 2);
#pragma unroll
                    for (int u = 0; u < 6; ++u) {
                        __builtin_amdgcn_sched_group_barrier(0x8, 1, 2);
                        __builtin_amdgcn_sched_group_barrier(0x2, 5, 2);
                    }
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 2);
                    __builtin_amdgcn_sched_group_barrier(0x8, 4, 2);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 2);
                    __builtin_amdgcn_sched_group_barrier(0x8, 2, 2);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 2);
                }
                if (i == 3 && (ks == 0 || ks == 2)) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 2, 1);
#pragma unroll
                    for (int u = 0; u < 2; ++u) {
                        __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
                        __builtin_amdgcn_sched_group_barrier(0x20, 1, 1);   // global -> LDS
                        __builtin_amdgcn_sched_group_barrier(0x8, 1, 1);
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        __builtin_amdgcn_sched_group_barrier(0x20, 1, 1);
                        __builtin_amdgcn_sched_group_barrier(0x8, 1, 1);
                    }
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
                    __builtin_amdgcn_sched_group_barrier(0x20, 1, 1);
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 1);
                    __builtin_amdgcn_sched_group_barrier(0x20, 2, 1);
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 1);
                    __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
                    __builtin_amdgcn_sched_group_barrier(0x8, 4, 1);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
                    __builtin_amdgcn_sched_group_barrier(0x8, 2, 1);
                    __builtin_amdgcn_sched_group_barrier(0x100, 2, 1);
                    __builtin_amdgcn_sched_group_barrier(0x8, 2, 1);
                    __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
                    __builtin_amdgcn_sched_group_barrier(0x8, 2, 1);
                    __builtin_amdgcn_sched_group_barrier(0x100, 3, 1);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (ks == 3) flush(3);
        }
    }
    __builtin_amdgcn_s_waitcnt(0);   // no load into LDS outlives the work-group

    double *C = F.Pi + (int64_t)w * N * N;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int q = q0 + 32 * wj + 16 * j + (lane & 15);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int p = p0 + 64 * wi + 16 * i + 4 * (lane >> 4) + r;
                if (p < N && q <= p) C[(int64_t)p * N + q] = acc[i][j][r];
            }
        }
}

int launch_syrk_bf16(brpa_ctx *ctx, const FragDev *fr, const int64_t *pre, int nfrag,
                     int64_t total) {
    if (total <= 0) return BRPA_OK;
    hipLaunchKernelGGL(k_syrk_bf16, dim3((unsigned)total), dim3(512), 0, ctx->stream, fr, pre,
                       nfrag);
    LAUNCH_CHECK(ctx);
    return BRPA_OK;
}
