// One output tile of an FP64 product on v_mfma_f64_16x16x4_f64 by a work-group of four
// waves (2 x 2): the loop of k_gemm_f64 and of the Cholesky's trailing update.
#pragma once
#include <type_traits>

#include "device_common.h"

constexpr int GKB = 16;    // k per LDS stage
typedef double d2_t __attribute__((ext_vector_type(2)));

// LDS layout of one operand's tile (ROWS rows, 128 or 64) and 16-k stage.  k-contiguous (KC): [row][k]
// with unpadded 16-double rows whose k pairs are XOR-swizzled by (row >> 1) & 7.
// Rows-contiguous: [k][row] with rows of DMA_KPR doubles (a pitch of 4 rows moves by
// half of the 64 LDS banks, so the four lane groups of a fragment read hit disjoint
// halves).
//
// A wave's loads, 16 bytes per lane (which need no more than the 4-byte alignment of every
// vector load, so odd leading dimensions take them too): KC the 8-row blocks ROWS / 4 w +
// 8 c, lane L the k pair (L % 8) ^ swizzle of row L / 8 of its block; rows-contiguous (128
// rows only) the k rows 4 w + c, lane L the rows 2 L, 2 L + 1.  The byte offsets from the
// tile's base at k = 0 (dma_base) are 32-bit (off_t), with leading dimensions of 2^21 or
// more (FAR) 64-bit, at the cost of their registers.
constexpr int DMA_KPR = 132;
template <bool KC>
constexpr int gemm_lds(int rows) {   // doubles of one stage
    return KC ? rows * GKB : GKB * DMA_KPR;
}
template <bool KC, int ROWS, bool FAR>
struct DmaSrc {
    static_assert(KC || ROWS == 128, "rows-contiguous operands have 128-row tiles");
    static constexpr int NLOAD = ROWS / 32;   // loads per wave and stage
    typedef std::conditional_t<FAR, uint64_t, uint32_t> off_t;
    off_t off[NLOAD];
};
template <bool KC, int ROWS, bool FAR>
__device__ __forceinline__ DmaSrc<KC, ROWS, FAR> dma_offsets(int64_t ldx, int r0, int rows, int wave,
                                                            int lane) {
    DmaSrc<KC, ROWS, FAR> s;
    typedef typename DmaSrc<KC, ROWS, FAR>::off_t off_t;
#pragma unroll
    for (int c = 0; c < s.NLOAD; ++c) {
        if (KC) {
            const int row = ROWS / 4 * wave + 8 * c + (lane >> 3);
            const int dk = 2 * ((lane & 7) ^ ((row >> 1) & 7));
            s.off[c] = 8u * ((off_t)ldx * (uint32_t)(min(r0 + row, rows - 1) - r0) + (uint32_t)dk);
        } else {
            // the pair of the last row of an odd count ends in the next k's first row
            // (dma_over)
            s.off[c] = 8u * ((uint32_t)(min(r0 + 2 * lane, (rows - 1) & ~1) - r0) +
                             (off_t)ldx * (uint32_t)(4 * wave + c));
        }
    }
    return s;
}
// whether a full stage that ends with the last k of all reads past the operand's end
template <bool KC, int ROWS>
__device__ __forceinline__ bool dma_over(int r0, int rows) {
    return !KC && (rows & 1) && r0 + ROWS > rows;
}
template <bool KC>
__device__ __forceinline__ const char *dma_base(const double *X, int64_t ldx, int r0) {
    return reinterpret_cast<const char *>(X + (KC ? ldx * r0 : (int64_t)r0));
}
// fragment of row `row` at the k pair 2 g4 + hh of a stage
template <bool KC>
__host__ __device__ __forceinline__ d2_t dma_frag(const double *L, int row, int g4, int hh) {
    if (KC) {
        const int kp = 2 * g4 + hh;
        return *reinterpret_cast<const d2_t *>(&L[row * GKB + 2 * (kp ^ ((row >> 1) & 7))]);
    }
    const int kr = 4 * g4 + 2 * hh;
    d2_t v;
    v.x = L[kr * DMA_KPR + row];
    v.y = L[(kr + 1) * DMA_KPR + row];
    return v;
}

// one operand's full stage at k0 into the LDS buffer L, straight from global memory
template <bool KC, int ROWS, bool FAR>
__device__ __forceinline__ void dma_stage(const char *base, const DmaSrc<KC, ROWS, FAR> &src, int64_t ldx,
                                          double *L, int wave, int k0) {
    // the builtin exists for the device pass only; the host pass never runs this
#if defined(__HIP_DEVICE_COMPILE__)
    typedef __attribute__((address_space(1))) const char gchar_t;
    typedef __attribute__((address_space(1))) const void gvoid_t;
    typedef __attribute__((address_space(3))) void lvoid_t;
    gchar_t *b = (gchar_t *)(base + 8 * (KC ? (int64_t)k0 : ldx * k0));
#pragma unroll
    for (int c = 0; c < src.NLOAD; ++c)
        __builtin_amdgcn_global_load_lds(
            (gvoid_t *)(b + src.off[c]),
            (lvoid_t *)(L + (KC ? (ROWS / 4 * wave + 8 * c) * GKB : (4 * wave + c) * DMA_KPR)), 16, 0, 0);
#endif
}
// the last stage when it has fewer than 16 k, or may not be read past its end: through
// registers, zeros past kend
template <bool KC, int ROWS>
__device__ __forceinline__ void dma_stage_tail(const double *__restrict__ X, int64_t ldx, int r0,
                                               int rows, double *L, int tid, int k0, int kend) {
#pragma unroll 1
    for (int u = 0; u < ROWS / 16; ++u) {
        const int e = tid + 256 * u;
        const int row = KC ? e >> 4 : e & 127, kk = KC ? e & 15 : e >> 7;
        const int64_t r = min(r0 + row, rows - 1);
        const double v = k0 + kk < kend ? X[KC ? k0 + kk + ldx * r : r + ldx * (k0 + kk)] : 0.0;
        L[KC ? row * GKB + 2 * ((kk >> 1) ^ ((row >> 1) & 7)) + (kk & 1) : kk * DMA_KPR + row] = v;
    }
}

// acc += rows m0 .. of op(A) times columns n0 .. of op(B) over k in [kbeg, kend) of [0, k): wave
// (wm, wn) = (wave / 2, wave % 2) holds the ROWS/2 x ROWS/2 block (wm, wn), acc[i][j][r]
// = element (16 i + lane % 16, 16 j + lane / 16 + 4 r) of it.  m, n: rows of the whole
// operands (past them the last row repeats).  FAR: 64-bit offsets.  Waves with active false only stage.  sA0/1, sB0/1: the two stages of each operand
// (gemm_lds doubles per stage).
//
// The fragments of either half of a stage are read while the other half is
// multiplied, one LDS read after each of the first MFMAs and then the loads of the
// coming stage after the next ones.  The barrier stands between the halves: by then
// the next stage has landed and every wave has read the current one, whose buffer
// takes the loads of the stage after the next.  Bound by MFMA issue: TN 8192 x 8192 x
// 2048 73.0 TFLOP/s, 4096^3 68.0, 4097^3 56 (50 with four bytes per lane for odd
// leading dimensions), 3072^2 x 4096 (whose last 64 of 576 tiles run one
// per CU) 52 (68.5, 64.0 and 38-46 with all reads, then all loads, ahead of the stage's
// MFMAs).
template <bool KCA, bool KCB, int ROWS, bool FAR = false>
__device__ __forceinline__ void gemm_tile(d4_t (&acc)[ROWS / 32][ROWS / 32],
                                          const double *__restrict__ A, int64_t lda, int m0, int m,
                                          const double *__restrict__ B, int64_t ldb, int n0, int n,
                                          int kbeg, int kend, int k, bool active, double *sA0,
                                          double *sA1, double *sB0, double *sB1) {
    constexpr int NB = ROWS / 32;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int rl = lane & 15, g4 = lane >> 4;
    const auto oa = dma_offsets<KCA, ROWS, FAR>(lda, m0, m, wave, lane);
    const auto ob = dma_offsets<KCB, ROWS, FAR>(ldb, n0, n, wave, lane);
    const char *ba = dma_base<KCA>(A, lda, m0), *bb = dma_base<KCB>(B, ldb, n0);
    const bool over = kend == k && (dma_over<KCA, ROWS>(m0, m) || dma_over<KCB, ROWS>(n0, n));
    const int nfull = (kend - kbeg - (over ? 1 : 0)) / GKB, ns = (kend - kbeg + GKB - 1) / GKB;
    auto stage = [&](int buf, int k0) {
        dma_stage(ba, oa, lda, buf ? sA1 : sA0, wave, k0);
        dma_stage(bb, ob, ldb, buf ? sB1 : sB0, wave, k0);
    };
    auto put = [&](int buf, int q) {
        if (q < nfull) {
            stage(buf, kbeg + GKB * q);
        } else if (q < ns) {
            dma_stage_tail<KCA, ROWS>(A, lda, m0, m, buf ? sA1 : sA0, tid, kbeg + GKB * q, kend);
            dma_stage_tail<KCB, ROWS>(B, ldb, n0, n, buf ? sB1 : sB0, tid, kbeg + GKB * q, kend);
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
    // one half of a stage: two k per lane
    auto frags = [&](d2_t (&a)[NB], d2_t (&b)[NB], int buf, int hh) {
#pragma unroll
        for (int i = 0; i < NB; ++i)
            a[i] = dma_frag<KCA>(buf ? sA1 : sA0, ROWS / 2 * wm + 16 * i + rl, g4, hh);
#pragma unroll
        for (int j = 0; j < NB; ++j)
            b[j] = dma_frag<KCB>(buf ? sB1 : sB0, ROWS / 2 * wn + 16 * j + rl, g4, hh);
    };
    auto mma = [&](const d2_t (&a)[NB], const d2_t (&b)[NB]) {
#pragma unroll
        for (int st = 0; st < 2; ++st)
#pragma unroll
            for (int i = 0; i < NB; ++i)
#pragma unroll
                for (int j = 0; j < NB; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[j][st], a[i][st], acc[i][j], 0,
                                                                     0, 0);
    };
    d2_t a0[NB], b0[NB], a1[NB], b1[NB];
    __syncthreads();
    put(1, 1);
    frags(a0, b0, 0, 0);
    constexpr int NM = 2 * NB * NB, NR = 2 * NB;      // MFMAs and LDS reads of a half
    constexpr int NL = 2 * (ROWS / 32);   // loads of a stage per wave
    constexpr int LG = NL < NM - NR ? NL : NM - NR;   // MFMAs they are spread over
    // with buf constant the compiler knows that a read of one stage does not wait for the loads
    // into the other
    auto step = [&](int buf, int q) {
        frags(a1, b1, buf, 1);
        mma(a0, b0);
#pragma unroll
        for (int u = 0; u < NR; ++u) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);     // MFMA
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // LDS read
        }
        __builtin_amdgcn_sched_group_barrier(0x8, NM - NR, 0);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        frags(a0, b0, buf ^ 1, 0);
        stage(buf, kbeg + GKB * (q + 2));
        mma(a1, b1);
#pragma unroll
        for (int u = 0; u < NR; ++u) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 1);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 1);
        }
#pragma unroll
        for (int u = 0; u < LG; ++u) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 1);
            __builtin_amdgcn_sched_group_barrier(0x20, (NL + LG - 1) / LG, 1);   // global -> LDS
        }
        __builtin_amdgcn_sched_group_barrier(0x8, NM - NR - LG, 1);
        __builtin_amdgcn_sched_barrier(0);
    };
    int q = 0;
    for (; q + 3 < nfull; q += 2) {
        step(0, q);
        step(1, q + 1);
    }
    int buf = 0;
    for (; q < ns; ++q, buf ^= 1) {
        frags(a1, b1, buf, 1);
        mma(a0, b0);
        if (q + 1 < ns) {
            __syncthreads();
            put(buf, q + 2);
            frags(a0, b0, buf ^ 1, 0);
        }
        mma(a1, b1);
    }
}
