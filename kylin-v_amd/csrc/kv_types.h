// Work descriptors shared by the host planners and the gfx950 kernels.  Plain data,
// no HIP types, so the planners build and run on any C++17 host compiler.
#pragma once

#include <cstdint>

namespace kv {

// ---- grouped complex GEMM ---------------------------------------------------------
// C_g[m,n] = alpha * sum_{s in segments of g} opA(A)_s[m,k] opB(B)_s[k,n]
// opA: 0 'N' A[m*lda+k], 1 'T' A[k*lda+m], 2 'C' conj(A[k*lda+m])
// opB: 0 'N' B[k*ldb+n], 1 'T' B[n*ldb+k], 2 'C' conj(B[n*ldb+k])
// C is row-major with leading dimension ldc.  Offsets count complex elements.
struct GemmSeg {
    int64_t a_off, b_off;
    int k, lda, ldb, pad;
};
struct GemmGroup {
    int64_t c_off;
    int m, n, ldc, seg_begin, seg_count, pad;
};
struct GemmTile {
    int group, tm, tn;
    int seg;  // the group's seg_begin: group and first segment load side by side
};

constexpr int GEMM_BM = 64, GEMM_BN = 64, GEMM_BK = 8;

// Tile shapes of the grouped GEMM (complex outputs per workgroup, K depth per LDS stage).
// Config 0 exists for every op pair; the others for the pairs on the hot path
// (NN, NT, CN, NC).
struct GemmConfig {
    int bm, bn, bk;
};
constexpr int kNumGemmConfigs = 7;
constexpr GemmConfig kGemmConfigs[kNumGemmConfigs] = {
    {64, 64, 8}, {64, 64, 16}, {128, 64, 8}, {64, 128, 8}, {128, 128, 8}, {128, 64, 16}, {64, 128, 16}};

// ---- MPO fold -----------------------------------------------------------------------
// out[out_base + p*out_pstride + q] = sum_t w_t * in[t.in_base + p*t.in_pstride + q]
// for p < P, q < Q.  A task with no terms writes zeros.
struct WTerm {
    int64_t in_base, in_pstride;
    double re, im;
};
struct WTask {
    int64_t out_base, out_pstride;
    int P, Q, term_begin, term_count;
};

// ---- two MPO folds as one: tasks expanded from the two folds' own lists ------------------
// A task of the second fold stands for S1 composite tasks (one per s1' of the first), whose
// terms are its own terms times those of the first fold's task that wrote the slice they read.
struct WComposeTask {
    int64_t out_base, out_pstride, s1_stride;  // of s1' = 0; out_base grows by s1_stride per s1'
    int64_t slot;                              // composite terms of s1' start at slot + s1' * maxt
    int P, Q, S1, task0;                       // composite tasks task0 .. task0 + S1 - 1
    int term_begin, term_count, maxt, pad;     // terms of the second fold
};
struct WComposeTerm {
    int64_t shift;  // added to the first fold's in_base
    double re, im;
    int f1_task, f1_stride;  // the first fold's task of s1' = 0 (-1: that slice is zero), per s1'
};

#ifdef __HIPCC__
#define KV_HD __host__ __device__
#else
#define KV_HD
#endif
// Composite task s1 of c into tasks[c.task0 + s1] and its terms.
KV_HD inline void wcompose_expand(const WComposeTask& c, int s1, const WComposeTerm* terms2, const WTask* tasks1,
                                  const WTerm* terms1, WTask* tasks, WTerm* terms) {
    WTask t;
    t.out_base = c.out_base + (int64_t)s1 * c.s1_stride;
    t.out_pstride = c.out_pstride;
    t.P = c.P;
    t.Q = c.Q;
    int64_t at = c.slot + (int64_t)s1 * c.maxt;
    t.term_begin = (int)at;
    for (int k2 = c.term_begin; k2 < c.term_begin + c.term_count; ++k2) {
        const WComposeTerm w2 = terms2[k2];
        if (w2.f1_task < 0) continue;
        const WTask t1 = tasks1[w2.f1_task + s1 * w2.f1_stride];
        for (int k1 = t1.term_begin; k1 < t1.term_begin + t1.term_count; ++k1) {
            const WTerm w1 = terms1[k1];
            WTerm w;
            w.in_base = w1.in_base + w2.shift;
            w.in_pstride = w1.in_pstride;
            w.re = w2.re * w1.re - w2.im * w1.im;
            w.im = w2.re * w1.im + w2.im * w1.re;
            terms[at++] = w;
        }
    }
    t.term_count = (int)(at - t.term_begin);
    tasks[c.task0 + s1] = t;
}

// ---- SVD of small sectors (launch_jacobi_svd) --------------------------------------------
constexpr int kJacobiMax = 64;  // largest smaller side

// ---- block permutation (tensor transpose) ----------------------------------------------
constexpr int PERM_MAXR = 6;
struct PermTask {
    int64_t in_off, out_off, size;
    int rank, pad;
    int oshape[PERM_MAXR];
    int64_t istride[PERM_MAXR];  // input stride of each OUTPUT axis
};

// ---- 2-D strided copies (sector gather / scatter for the SVD) -------------------------
// dst[dst_off + r*dst_ld + c] = f * src[src_off + r*src_ld + c], f = 1, s[scale_off+r]
// (scale_mode 1) or s[scale_off+c] (scale_mode 2).
struct Copy2D {
    int64_t src_off, dst_off;
    int rows, cols, src_ld, dst_ld, scale_mode, scale_off;
};

// ---- overlap over matching block pairs ------------------------------------------------
// sum over pairs of conj(x[x_off + e]) y[y_off + e], e < size
struct DotPair {
    int64_t x_off, y_off, size;
};

}  // namespace kv
