// gfx950 (CDNA4) kernels of the Holstein TDVP engine.
//
//  * zgemm_grouped: complex GEMM over a device-resident list of U(1) block pairs.  One
//    launch covers every output block of a contraction stage; a group sums its K
//    segments (the block pairs that land on the same output block) inside one tile,
//    so there are no atomics and results are deterministic.  Complex products run as
//    four real MFMAs (re.re - im.im, re.im + im.re) on v_mfma_f64_16x16x4f64, and in
//    FP32 as three (re.re, im.im, (re+im)(re+im): Gauss's product) on
//    v_mfma_f32_16x16x4f32; 64x64 complex tile per 256-thread workgroup, 4 waves in
//    a 2x2 arrangement of 32x32 complex wave tiles, operands staged through LDS.
//  * wfold: applies the sparse MPO tensor as a gather-sum over contiguous slices.
//  * perm / copy2d: block transposes and sector gather/scatter.
//  * FP64 vector algebra for the Lanczos recurrence (deterministic two-pass reductions).
#include <mutex>

#include "kv_kernels.h"
#include "kv_runtime.h"

namespace kv {

typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// ---- sums over a wave's lanes by DPP moves and lane swaps (a few cycles a step; a permute through
// LDS takes about a hundred) ---------------------------------------------------------------
// v[t + 32], v[t + 16]: valid in lanes 0..31 / in the lanes of each even row of 16
__device__ inline double lane_up32(double v) {
    const long long b = __double_as_longlong(v);
    const auto lo = __builtin_amdgcn_permlane32_swap((int)b, (int)b, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((int)(b >> 32), (int)(b >> 32), false, false);
    return __longlong_as_double(((long long)hi[1] << 32) | (unsigned)lo[1]);
}
__device__ inline double lane_up16(double v) {
    const long long b = __double_as_longlong(v);
    const auto lo = __builtin_amdgcn_permlane16_swap((int)b, (int)b, false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap((int)(b >> 32), (int)(b >> 32), false, false);
    return __longlong_as_double(((long long)hi[1] << 32) | (unsigned)lo[1]);
}
// a DPP move of both halves: CTRL 0x100 + s shifts a row of 16 so that lane t reads lane t + s,
// 0xB1 / 0x4E swap neighbours / pairs, 0x141 mirrors rows of 8, 0x140 rows of 16
template <int CTRL>
__device__ inline double lane_dpp(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)b, CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), CTRL, 0xF, 0xF, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ inline double lane_first(double v) {  // lane 0's value in every lane
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readfirstlane((int)b), hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
// The pairwise tree v[t] += v[t + s], s = 32, 16, ..., 1: lane 0 holds the total.
__device__ inline double tree64(double v) {
    v += lane_up32(v);
    v += lane_up16(v);
    v += lane_dpp<0x108>(v);
    v += lane_dpp<0x104>(v);
    v += lane_dpp<0x102>(v);
    v += lane_dpp<0x101>(v);
    return v;
}
// The sum over each row of 16 in all of its lanes.
__device__ inline double row_all(double v) {
    v += lane_dpp<0xB1>(v);
    v += lane_dpp<0x4E>(v);
    v += lane_dpp<0x141>(v);
    v += lane_dpp<0x140>(v);
    return v;
}

// The device's wall clock (100 MHz) at the start of a launch's first workgroup.
__device__ inline void write_mark(Mark* mark) {
    if (mark && (blockIdx.x | blockIdx.y | threadIdx.x) == 0) *mark = wall_clock64();
}
__global__ void mark_kernel(Mark* mark) { write_mark(mark); }
void launch_mark(hipStream_t st, Mark* mark) {
    hipLaunchKernelGGL(mark_kernel, dim3(1), dim3(1), 0, st, mark);
    KV_HIP(hipGetLastError());
}

template <class T> struct Cx;
template <> struct Cx<double> {
    using T2 = double2;
    using acc = f64x4;
    __device__ static inline acc mfma(double a, double b, acc c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    // v_mfma_f64_16x16x4f64: lane l, accumulator item v holds D[l/16 + 4v][l%16]
    // (measured on gfx950 with one-hot operands)
    __device__ static inline int out_row(int lk, int v) { return lk + 4 * v; }
};
template <> struct Cx<float> {
    using T2 = float2;
    using acc = f32x4;
    __device__ static inline acc mfma(float a, float b, acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    // v_mfma_f32_16x16x4f32: lane l, accumulator item v holds D[4(l/16) + v][l%16]
    __device__ static inline int out_row(int lk, int v) { return 4 * lk + v; }
};

template <class T2> struct ScalarOf;
template <> struct ScalarOf<double2> { using T = double; };
template <> struct ScalarOf<float2> { using T = float; };

// ------------------------------------------------------------------------------------
// grouped complex GEMM
// ------------------------------------------------------------------------------------
// Tile BM x BN complex outputs per 256-thread workgroup; 4 waves in a 2x2 arrangement, each
// owning (BM/2) x (BN/2) outputs as 16x16 MFMA sub-tiles; BK complex K per LDS stage.
// Workgroup i runs tile i.  Workgroups are dispatched round-robin over the 8 XCDs and the
// tile list is row-major per group, so tiles that share a B panel (same tile column, rows
// a multiple of 8 tiles apart when the tile-column count is) land on one XCD's L2; a
// remap giving each XCD a contiguous run of tiles measured 20% slower on the H_eff stages.
template <class T, int OPA, int OPB, int BM, int BN, int BK>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(BM * BN <= 4096 ? 3 : 1))) void zgemm_grouped_kernel(
    const typename Cx<T>::T2* __restrict__ A, const typename Cx<T>::T2* __restrict__ B,
    typename Cx<T>::T2* __restrict__ C, const GemmTile* __restrict__ tiles,
    const GemmGroup* __restrict__ groups, const GemmSeg* __restrict__ segs, T alpha_re,
    T alpha_im, const int* __restrict__ stop, Mark* mark) {
    if (stop && *stop) return;
    write_mark(mark);
    using T2 = typename Cx<T>::T2;
    using acc_t = typename Cx<T>::acc;
    constexpr int SI = BM / 32, SJ = BN / 32;  // 16x16 sub-tiles per wave
    __shared__ T2 As[2][BK][BM + 1];  // double-buffered: one barrier per K stage
    __shared__ T2 Bs[2][BK][BN + 1];

    const GemmTile tile = tiles[blockIdx.x];
    const GemmGroup g = groups[tile.group];
    const int m0 = tile.tm * BM, n0 = tile.tn * BN;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
    const int lr = lane & 15, lk = lane >> 4;

    // FP64: cre = sum re.re - im.im, cim = sum re.im + im.re (four MFMAs per step).
    // FP32: three MFMAs per step (Gauss): cre = sum re.re, cp2 = sum im.im,
    // cim = sum (re + im)(re + im); the epilogue forms re = cre - cp2, im = cim - cre - cp2.
    constexpr bool kGauss = sizeof(T) == sizeof(float);
    acc_t cre[SI][SJ], cim[SI][SJ], cp2[SI][SJ];
#pragma unroll
    for (int i = 0; i < SI; ++i)
#pragma unroll
        for (int j = 0; j < SJ; ++j) {
            cre[i][j] = acc_t{0, 0, 0, 0};
            cim[i][j] = acc_t{0, 0, 0, 0};
            cp2[i][j] = acc_t{0, 0, 0, 0};
        }

    // K stages run over (segment, k0) pairs.  The next stage's operands are loaded into
    // registers while the current one is multiplied out of LDS, so global latency hides
    // behind the MFMAs of the same workgroup.
    constexpr int NA = (BM * BK) / 256, NB = (BN * BK) / 256;
    T2 ra[NA], rb[NB];
    // FP32 complex operands load two neighbours along each operand's contiguous index per
    // thread (one 16-byte access when the segment's offset and leading dimension are even).
    constexpr bool kPair = sizeof(T2) == 8;
    auto load = [&](int s, int k0) {
        const GemmSeg sg = segs[tile.seg + s];
        const T2* __restrict__ a = A + sg.a_off;
        const T2* __restrict__ b = B + sg.b_off;
        const int K = sg.k;
        if constexpr (kPair) {
            const bool alA = ((sg.a_off | (int64_t)sg.lda) & 1) == 0;
            const bool alB = ((sg.b_off | (int64_t)sg.ldb) & 1) == 0;
#pragma unroll
            for (int r = 0; r < NA / 2; ++r) {
                const int e = tid + r * 256;
                const int mm = (OPA == 0) ? e / (BK / 2) : 2 * (e % (BM / 2));
                const int kk = (OPA == 0) ? 2 * (e % (BK / 2)) : e / (BM / 2);
                const int gm = m0 + mm, gk = k0 + kk;
                T2 v0, v1;
                v0.x = 0;
                v0.y = 0;
                v1 = v0;
                if (OPA == 0) {  // neighbours along k
                    if (gm < g.m) {
                        const T2* pa = a + (int64_t)gm * sg.lda + gk;
                        if (alA && gk + 1 < K) {
                            const float4 q = *reinterpret_cast<const float4*>(pa);
                            v0.x = q.x;
                            v0.y = q.y;
                            v1.x = q.z;
                            v1.y = q.w;
                        } else {
                            if (gk < K) v0 = pa[0];
                            if (gk + 1 < K) v1 = pa[1];
                        }
                    }
                } else {  // neighbours along m
                    if (gk < K) {
                        const T2* pa = a + (int64_t)gk * sg.lda + gm;
                        if (alA && gm + 1 < g.m) {
                            const float4 q = *reinterpret_cast<const float4*>(pa);
                            v0.x = q.x;
                            v0.y = q.y;
                            v1.x = q.z;
                            v1.y = q.w;
                        } else {
                            if (gm < g.m) v0 = pa[0];
                            if (gm + 1 < g.m) v1 = pa[1];
                        }
                    }
                }
                if (OPA == 2) {
                    v0.y = -v0.y;
                    v1.y = -v1.y;
                }
                ra[2 * r] = v0;
                ra[2 * r + 1] = v1;
            }
#pragma unroll
            for (int r = 0; r < NB / 2; ++r) {
                const int e = tid + r * 256;
                const int nn = (OPB == 0) ? 2 * (e % (BN / 2)) : e / (BK / 2);
                const int kk = (OPB == 0) ? e / (BN / 2) : 2 * (e % (BK / 2));
                const int gn = n0 + nn, gk = k0 + kk;
                T2 v0, v1;
                v0.x = 0;
                v0.y = 0;
                v1 = v0;
                if (OPB == 0) {  // neighbours along n
                    if (gk < K) {
                        const T2* pb = b + (int64_t)gk * sg.ldb + gn;
                        if (alB && gn + 1 < g.n) {
                            const float4 q = *reinterpret_cast<const float4*>(pb);
                            v0.x = q.x;
                            v0.y = q.y;
                            v1.x = q.z;
                            v1.y = q.w;
                        } else {
                            if (gn < g.n) v0 = pb[0];
                            if (gn + 1 < g.n) v1 = pb[1];
                        }
                    }
                } else {  // neighbours along k
                    if (gn < g.n) {
                        const T2* pb = b + (int64_t)gn * sg.ldb + gk;
                        if (alB && gk + 1 < K) {
                            const float4 q = *reinterpret_cast<const float4*>(pb);
                            v0.x = q.x;
                            v0.y = q.y;
                            v1.x = q.z;
                            v1.y = q.w;
                        } else {
                            if (gk < K) v0 = pb[0];
                            if (gk + 1 < K) v1 = pb[1];
                        }
                    }
                }
                if (OPB == 2) {
                    v0.y = -v0.y;
                    v1.y = -v1.y;
                }
                rb[2 * r] = v0;
                rb[2 * r + 1] = v1;
            }
            return;
        }
#pragma unroll
        for (int r = 0; r < NA; ++r) {
            const int e = tid + r * 256;
            int mm, kk;
            if (OPA == 0) {
                mm = e / BK;
                kk = e % BK;
            } else {
                kk = e / BM;
                mm = e % BM;
            }
            const int gm = m0 + mm, gk = k0 + kk;
            T2 v;
            v.x = 0;
            v.y = 0;
            if (gm < g.m && gk < K) {
                v = (OPA == 0) ? a[(int64_t)gm * sg.lda + gk] : a[(int64_t)gk * sg.lda + gm];
                if (OPA == 2) v.y = -v.y;
            }
            ra[r] = v;
        }
#pragma unroll
        for (int r = 0; r < NB; ++r) {
            const int e = tid + r * 256;
            int nn, kk;
            if (OPB == 0) {
                kk = e / BN;
                nn = e % BN;
            } else {
                nn = e / BK;
                kk = e % BK;
            }
            const int gn = n0 + nn, gk = k0 + kk;
            T2 v;
            v.x = 0;
            v.y = 0;
            if (gn < g.n && gk < K) {
                v = (OPB == 0) ? b[(int64_t)gk * sg.ldb + gn] : b[(int64_t)gn * sg.ldb + gk];
                if (OPB == 2) v.y = -v.y;
            }
            rb[r] = v;
        }
    };
    auto store = [&](int buf) {
        if constexpr (kPair) {
#pragma unroll
            for (int r = 0; r < NA / 2; ++r) {
                const int e = tid + r * 256;
                const int mm = (OPA == 0) ? e / (BK / 2) : 2 * (e % (BM / 2));
                const int kk = (OPA == 0) ? 2 * (e % (BK / 2)) : e / (BM / 2);
                As[buf][kk][mm] = ra[2 * r];
                if (OPA == 0)
                    As[buf][kk + 1][mm] = ra[2 * r + 1];
                else
                    As[buf][kk][mm + 1] = ra[2 * r + 1];
            }
#pragma unroll
            for (int r = 0; r < NB / 2; ++r) {
                const int e = tid + r * 256;
                const int nn = (OPB == 0) ? 2 * (e % (BN / 2)) : e / (BK / 2);
                const int kk = (OPB == 0) ? e / (BN / 2) : 2 * (e % (BK / 2));
                Bs[buf][kk][nn] = rb[2 * r];
                if (OPB == 0)
                    Bs[buf][kk][nn + 1] = rb[2 * r + 1];
                else
                    Bs[buf][kk + 1][nn] = rb[2 * r + 1];
            }
            return;
        }
#pragma unroll
        for (int r = 0; r < NA; ++r) {
            const int e = tid + r * 256;
            const int mm = (OPA == 0) ? e / BK : e % BM;
            const int kk = (OPA == 0) ? e % BK : e / BM;
            As[buf][kk][mm] = ra[r];
        }
#pragma unroll
        for (int r = 0; r < NB; ++r) {
            const int e = tid + r * 256;
            const int nn = (OPB == 0) ? e % BN : e / BK;
            const int kk = (OPB == 0) ? e / BN : e % BK;
            Bs[buf][kk][nn] = rb[r];
        }
    };
    int s = 0, k0 = 0, buf = 0;
    while (s < g.seg_count && segs[tile.seg + s].k <= 0) ++s;
    if (s < g.seg_count) {
        load(s, 0);
        store(0);
    }
    __syncthreads();
    // iteration t multiplies out of buffer buf while the operands of stage t+1 go into the
    // other one; the single barrier ends both (the other buffer was last read in t-1)
    while (s < g.seg_count) {
        int s2 = s, k2 = k0 + BK;
        if (k2 >= segs[tile.seg + s].k) {
            k2 = 0;
            ++s2;
            while (s2 < g.seg_count && segs[tile.seg + s2].k <= 0) ++s2;
        }
        if (s2 < g.seg_count) load(s2, k2);
#pragma unroll
        for (int kq = 0; kq < BK; kq += 4) {
            T2 av[SI], bv[SJ];
#pragma unroll
            for (int i = 0; i < SI; ++i) av[i] = As[buf][kq + lk][wm + i * 16 + lr];
#pragma unroll
            for (int j = 0; j < SJ; ++j) bv[j] = Bs[buf][kq + lk][wn + j * 16 + lr];
            if constexpr (kGauss) {
                T as[SI], bs[SJ];
#pragma unroll
                for (int i = 0; i < SI; ++i) as[i] = av[i].x + av[i].y;
#pragma unroll
                for (int j = 0; j < SJ; ++j) bs[j] = bv[j].x + bv[j].y;
#pragma unroll
                for (int i = 0; i < SI; ++i)
#pragma unroll
                    for (int j = 0; j < SJ; ++j) {
                        cre[i][j] = Cx<T>::mfma(av[i].x, bv[j].x, cre[i][j]);
                        cp2[i][j] = Cx<T>::mfma(av[i].y, bv[j].y, cp2[i][j]);
                        cim[i][j] = Cx<T>::mfma(as[i], bs[j], cim[i][j]);
                    }
            } else {
#pragma unroll
                for (int i = 0; i < SI; ++i)
#pragma unroll
                    for (int j = 0; j < SJ; ++j) {
                        cre[i][j] = Cx<T>::mfma(av[i].x, bv[j].x, cre[i][j]);
                        cre[i][j] = Cx<T>::mfma(-av[i].y, bv[j].y, cre[i][j]);
                        cim[i][j] = Cx<T>::mfma(av[i].x, bv[j].y, cim[i][j]);
                        cim[i][j] = Cx<T>::mfma(av[i].y, bv[j].x, cim[i][j]);
                    }
            }
        }
        if (s2 < g.seg_count) store(buf ^ 1);
        __syncthreads();
        buf ^= 1;
        s = s2;
        k0 = k2;
    }
    // epilogue: MFMA output layout per type (Cx<T>::out_row)
#pragma unroll
    for (int i = 0; i < SI; ++i)
#pragma unroll
        for (int j = 0; j < SJ; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = m0 + wm + i * 16 + Cx<T>::out_row(lk, v);
                const int col = n0 + wn + j * 16 + lr;
                if (row < g.m && col < g.n) {
                    T re = cre[i][j][v], im = cim[i][j][v];
                    if constexpr (kGauss) {
                        const T p1 = re, p2 = cp2[i][j][v];
                        re = p1 - p2;
                        im = im - p1 - p2;
                    }
                    T2 o;
                    o.x = alpha_re * re - alpha_im * im;
                    o.y = alpha_re * im + alpha_im * re;
                    C[g.c_off + (int64_t)row * g.ldc + col] = o;
                }
            }
}

template <class T2>
void launch_gemm(hipStream_t st, int opA, int opB, const T2* A, const T2* B, T2* C,
                 const GemmTile* tiles, int ntiles, const GemmGroup* groups,
                 const GemmSeg* segs, double alpha_re, double alpha_im, int cfg, const int* stop,
                 Mark* mark) {
    using T = typename ScalarOf<T2>::T;
    if (ntiles <= 0) return;
    const dim3 grid(ntiles), block(256);
    const T ar = (T)alpha_re, ai = (T)alpha_im;
#define KV_GEMM_CASE(C_, OA, OB, BM_, BN_, BK_)                                                  \
    if (cfg == C_ && opA == OA && opB == OB) {                                                 \
        hipLaunchKernelGGL((zgemm_grouped_kernel<T, OA, OB, BM_, BN_, BK_>), grid, block, 0, st, \
                           A, B, C, tiles, groups, segs, ar, ai, stop, mark);                  \
        KV_HIP(hipGetLastError());                                                             \
        return;                                                                                \
    }
#define KV_GEMM_ALL_OPS(C_, BM_, BN_, BK_)  \
    KV_GEMM_CASE(C_, 0, 0, BM_, BN_, BK_)   \
    KV_GEMM_CASE(C_, 0, 1, BM_, BN_, BK_)   \
    KV_GEMM_CASE(C_, 0, 2, BM_, BN_, BK_)   \
    KV_GEMM_CASE(C_, 1, 0, BM_, BN_, BK_)   \
    KV_GEMM_CASE(C_, 1, 1, BM_, BN_, BK_)   \
    KV_GEMM_CASE(C_, 1, 2, BM_, BN_, BK_)   \
    KV_GEMM_CASE(C_, 2, 0, BM_, BN_, BK_)   \
    KV_GEMM_CASE(C_, 2, 1, BM_, BN_, BK_)   \
    KV_GEMM_CASE(C_, 2, 2, BM_, BN_, BK_)
#define KV_GEMM_HOT_OPS(C_, BM_, BN_, BK_)  \
    KV_GEMM_CASE(C_, 0, 0, BM_, BN_, BK_)   \
    KV_GEMM_CASE(C_, 0, 1, BM_, BN_, BK_)   \
    KV_GEMM_CASE(C_, 2, 0, BM_, BN_, BK_)   \
    KV_GEMM_CASE(C_, 0, 2, BM_, BN_, BK_)
    KV_GEMM_ALL_OPS(0, 64, 64, 8)
    KV_GEMM_HOT_OPS(1, 64, 64, 16)
    KV_GEMM_HOT_OPS(2, 128, 64, 8)
    KV_GEMM_HOT_OPS(3, 64, 128, 8)
    if constexpr (sizeof(T) == sizeof(float)) {  // the FP64 128x128 tile spills registers
        KV_GEMM_HOT_OPS(4, 128, 128, 8)
    }
    KV_GEMM_HOT_OPS(5, 128, 64, 16)
    KV_GEMM_HOT_OPS(6, 64, 128, 16)
#undef KV_GEMM_HOT_OPS
#undef KV_GEMM_ALL_OPS
#undef KV_GEMM_CASE
    if (cfg != 0) {  // op pair without a specialised tile: fall back to the 64x64 tile
        throw Error(ERR_INTERNAL, "launch_gemm: tile config not built for this op pair");
    }
    throw Error(ERR_ARG, "launch_gemm: bad op codes");
}

bool gemm_config_supports(int cfg, int opA, int opB, bool fp64) {
    if (cfg == 0) return opA >= 0 && opA <= 2 && opB >= 0 && opB <= 2;
    if (cfg == 4 && fp64) return false;
    return (opA == 0 && opB == 0) || (opA == 0 && opB == 1) || (opA == 2 && opB == 0) ||
           (opA == 0 && opB == 2);
}

template void launch_gemm<double2>(hipStream_t, int, int, const double2*, const double2*,
                                   double2*, const GemmTile*, int, const GemmGroup*,
                                   const GemmSeg*, double, double, int, const int*, Mark*);
template void launch_gemm<float2>(hipStream_t, int, int, const float2*, const float2*,
                                  float2*, const GemmTile*, int, const GemmGroup*,
                                  const GemmSeg*, double, double, int, const int*, Mark*);

// ------------------------------------------------------------------------------------
// grouped complex GEMM, split-BF16 (FP32 operands and accumulation)
// ------------------------------------------------------------------------------------
// Every FP32 operand x is split into x_hi = bf16(x) and x_lo = bf16(x - x_hi) while it is
// staged into LDS; a real product is x_hi*y_hi + x_hi*y_lo + x_lo*y_hi on
// v_mfma_f32_16x16x32_bf16 (the lo*lo term, ~2^-16 relative, is dropped).  A complex
// product is four real products, i.e. 12 MFMAs per 16x16x32 complex step.  Same tiles,
// groups and K segments as zgemm_grouped_kernel.
// LDS holds each operand as four planes (re_hi, re_lo, im_hi, im_lo), K contiguous per row
// of A and per column of B, so a lane's eight K values are one 16-byte LDS read:
// v_mfma_f32_16x16x32_bf16 lane l takes A[l%16][8(l/16)..8(l/16)+7] and
// B[8(l/16)..8(l/16)+7][l%16]; accumulator item v holds D[4(l/16)+v][l%16].
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));

__device__ inline void split2(float x0, float x1, bf16x2& hi, bf16x2& lo) {
    const __bf16 h0 = (__bf16)x0, h1 = (__bf16)x1;
    hi = bf16x2{h0, h1};
    lo = bf16x2{(__bf16)(x0 - (float)h0), (__bf16)(x1 - (float)h1)};
}

// NT threads = 64 * (BM / (16 SI)) * (BN / (16 SJ)); each wave owns SI x SJ sub-tiles of
// 16x16 outputs.  The im.im product is accumulated with the B imaginary planes sign-
// flipped (exact in bf16), so each sub-tile keeps two accumulators (re, im).
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));

__device__ inline bf16x8 bf16_neg(bf16x8 v) {
    return __builtin_bit_cast(bf16x8, __builtin_bit_cast(u16x8, v) ^ (u16x8)(unsigned short)0x8000);
}

template <int OPA, int OPB, int BM, int BN, int SI, int SJ>
__global__ __launch_bounds__(64 * (BM / (16 * SI)) * (BN / (16 * SJ))) void zgemm_bf16x3_kernel(
    const float2* __restrict__ A, const float2* __restrict__ B, float2* __restrict__ C,
    const GemmTile* __restrict__ tiles, const GemmGroup* __restrict__ groups,
    const GemmSeg* __restrict__ segs, float alpha_re, float alpha_im, const int* __restrict__ stop,
    Mark* mark) {
    if (stop && *stop) return;
    write_mark(mark);
    constexpr int BK = 32, LDK = BK + 8;  // row pitch stays a multiple of 16 bytes
    constexpr int WN = BN / (16 * SJ), NT = 64 * (BM / (16 * SI)) * WN;
    __shared__ __attribute__((aligned(16))) __bf16 As[4][BM][LDK];
    __shared__ __attribute__((aligned(16))) __bf16 Bs[4][BN][LDK];

    const GemmTile tile = tiles[blockIdx.x];
    const GemmGroup g = groups[tile.group];
    const int m0 = tile.tm * BM, n0 = tile.tn * BN;
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int wm = (wave / WN) * (16 * SI), wn = (wave % WN) * (16 * SJ);
    const int lr = lane & 15, lk = lane >> 4;

    f32x4 cre[SI][SJ], cim[SI][SJ];
#pragma unroll
    for (int i = 0; i < SI; ++i)
#pragma unroll
        for (int j = 0; j < SJ; ++j) {
            cre[i][j] = f32x4{0, 0, 0, 0};
            cim[i][j] = f32x4{0, 0, 0, 0};
        }

    // K stages run over (segment, k0) pairs.  The raw FP32 operands of the next stage are
    // loaded into registers while the current one is multiplied out of LDS; they are split
    // into the bf16 planes and stored once every wave has finished reading.
    constexpr int RA = (BM * BK / 2) / NT, RB = (BN * BK / 2) / NT;
    float2 ra[RA][2], rb[RB][2];
    auto load = [&](int s, int k0) {
        const GemmSeg sg = segs[tile.seg + s];
        const float2* __restrict__ a = A + sg.a_off;
        const float2* __restrict__ b = B + sg.b_off;
        const int K = sg.k;
#pragma unroll
        for (int r = 0; r < RA; ++r) {
            const int e = tid + r * NT;
            int mm, kk;
            if (OPA == 0) {
                mm = e / (BK / 2);
                kk = 2 * (e % (BK / 2));
            } else {
                mm = e % BM;
                kk = 2 * (e / BM);
            }
            const int gm = m0 + mm, gk = k0 + kk;
            float2 v0 = make_float2(0.f, 0.f), v1 = make_float2(0.f, 0.f);
            if (gm < g.m) {
                if (OPA == 0) {
                    const float2* row = a + (int64_t)gm * sg.lda;
                    if (gk < K) v0 = row[gk];
                    if (gk + 1 < K) v1 = row[gk + 1];
                } else {
                    if (gk < K) v0 = a[(int64_t)gk * sg.lda + gm];
                    if (gk + 1 < K) v1 = a[(int64_t)(gk + 1) * sg.lda + gm];
                }
            }
            if (OPA == 2) {
                v0.y = -v0.y;
                v1.y = -v1.y;
            }
            ra[r][0] = v0;
            ra[r][1] = v1;
        }
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            const int e = tid + r * NT;
            int nn, kk;
            if (OPB == 0) {
                nn = e % BN;
                kk = 2 * (e / BN);
            } else {
                nn = e / (BK / 2);
                kk = 2 * (e % (BK / 2));
            }
            const int gn = n0 + nn, gk = k0 + kk;
            float2 v0 = make_float2(0.f, 0.f), v1 = make_float2(0.f, 0.f);
            if (gn < g.n) {
                if (OPB == 0) {
                    if (gk < K) v0 = b[(int64_t)gk * sg.ldb + gn];
                    if (gk + 1 < K) v1 = b[(int64_t)(gk + 1) * sg.ldb + gn];
                } else {
                    const float2* col = b + (int64_t)gn * sg.ldb;
                    if (gk < K) v0 = col[gk];
                    if (gk + 1 < K) v1 = col[gk + 1];
                }
            }
            if (OPB == 2) {
                v0.y = -v0.y;
                v1.y = -v1.y;
            }
            rb[r][0] = v0;
            rb[r][1] = v1;
        }
    };
    auto store = [&] {
#pragma unroll
        for (int r = 0; r < RA; ++r) {
            const int e = tid + r * NT;
            const int mm = (OPA == 0) ? e / (BK / 2) : e % BM;
            const int kk = (OPA == 0) ? 2 * (e % (BK / 2)) : 2 * (e / BM);
            bf16x2 h, l;
            split2(ra[r][0].x, ra[r][1].x, h, l);
            *(bf16x2*)&As[0][mm][kk] = h;
            *(bf16x2*)&As[1][mm][kk] = l;
            split2(ra[r][0].y, ra[r][1].y, h, l);
            *(bf16x2*)&As[2][mm][kk] = h;
            *(bf16x2*)&As[3][mm][kk] = l;
        }
#pragma unroll
        for (int r = 0; r < RB; ++r) {
            const int e = tid + r * NT;
            const int nn = (OPB == 0) ? e % BN : e / (BK / 2);
            const int kk = (OPB == 0) ? 2 * (e / BN) : 2 * (e % (BK / 2));
            bf16x2 h, l;
            split2(rb[r][0].x, rb[r][1].x, h, l);
            *(bf16x2*)&Bs[0][nn][kk] = h;
            *(bf16x2*)&Bs[1][nn][kk] = l;
            split2(rb[r][0].y, rb[r][1].y, h, l);
            *(bf16x2*)&Bs[2][nn][kk] = h;
            *(bf16x2*)&Bs[3][nn][kk] = l;
        }
    };
    int s = 0, k0 = 0;
    while (s < g.seg_count && segs[tile.seg + s].k <= 0) ++s;
    if (s < g.seg_count) {
        load(s, 0);
        store();
    }
    __syncthreads();
    while (s < g.seg_count) {
        int s2 = s, k2 = k0 + BK;
        if (k2 >= segs[tile.seg + s].k) {
            k2 = 0;
            ++s2;
            while (s2 < g.seg_count && segs[tile.seg + s2].k <= 0) ++s2;
        }
        if (s2 < g.seg_count) load(s2, k2);
        {
            bf16x8 af[SI][4], bf[SJ][4], bn[SJ][2];
#pragma unroll
            for (int i = 0; i < SI; ++i)
#pragma unroll
                for (int p = 0; p < 4; ++p)
                    af[i][p] = *(const bf16x8*)&As[p][wm + i * 16 + lr][8 * lk];
#pragma unroll
            for (int j = 0; j < SJ; ++j) {
#pragma unroll
                for (int p = 0; p < 4; ++p)
                    bf[j][p] = *(const bf16x8*)&Bs[p][wn + j * 16 + lr][8 * lk];
                bn[j][0] = bf16_neg(bf[j][2]);
                bn[j][1] = bf16_neg(bf[j][3]);
            }
#pragma unroll
            for (int i = 0; i < SI; ++i)
#pragma unroll
                for (int j = 0; j < SJ; ++j) {
                    f32x4 re = cre[i][j], im = cim[i][j];
                    re = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i][0], bf[j][0], re, 0, 0, 0);
                    re = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i][0], bf[j][1], re, 0, 0, 0);
                    re = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i][1], bf[j][0], re, 0, 0, 0);
                    re = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i][2], bn[j][0], re, 0, 0, 0);
                    re = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i][2], bn[j][1], re, 0, 0, 0);
                    re = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i][3], bn[j][0], re, 0, 0, 0);
                    im = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i][0], bf[j][2], im, 0, 0, 0);
                    im = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i][0], bf[j][3], im, 0, 0, 0);
                    im = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i][1], bf[j][2], im, 0, 0, 0);
                    im = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i][2], bf[j][0], im, 0, 0, 0);
                    im = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i][2], bf[j][1], im, 0, 0, 0);
                    im = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[i][3], bf[j][0], im, 0, 0, 0);
                    cre[i][j] = re;
                    cim[i][j] = im;
                }
        }
        __syncthreads();  // every wave has read this stage's planes
        if (s2 < g.seg_count) {
            store();
            __syncthreads();
        }
        s = s2;
        k0 = k2;
    }
#pragma unroll
    for (int i = 0; i < SI; ++i)
#pragma unroll
        for (int j = 0; j < SJ; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int row = m0 + wm + i * 16 + 4 * lk + v;
                const int col = n0 + wn + j * 16 + lr;
                if (row < g.m && col < g.n) {
                    const float re = cre[i][j][v], im = cim[i][j][v];
                    float2 o;
                    o.x = alpha_re * re - alpha_im * im;
                    o.y = alpha_re * im + alpha_im * re;
                    C[g.c_off + (int64_t)row * g.ldc + col] = o;
                }
            }
}

// cfg 0: 64x64 tile (256 threads); cfg 4: 128x128 tile (512 threads), same tile lists as
// the FP32 kernel's configs 0 and 4.
void launch_gemm_bf16x3(hipStream_t st, int opA, int opB, const float2* A, const float2* B,
                        float2* C, const GemmTile* tiles, int ntiles, const GemmGroup* groups,
                        const GemmSeg* segs, double alpha_re, double alpha_im, int cfg, const int* stop,
                 Mark* mark) {
    if (ntiles <= 0) return;
    const float ar = (float)alpha_re, ai = (float)alpha_im;
#define KV_BF_CASE(OA, OB)                                                                     \
    if (opA == OA && opB == OB) {                                                              \
        if (cfg == 4)                                                                          \
            hipLaunchKernelGGL((zgemm_bf16x3_kernel<OA, OB, 128, 128, 4, 2>), dim3(ntiles),     \
                               dim3(512), 0, st, A, B, C, tiles, groups, segs, ar, ai, stop, mark); \
        else                                                                                   \
            hipLaunchKernelGGL((zgemm_bf16x3_kernel<OA, OB, 64, 64, 2, 2>), dim3(ntiles),       \
                               dim3(256), 0, st, A, B, C, tiles, groups, segs, ar, ai, stop, mark); \
        KV_HIP(hipGetLastError());                                                             \
        return;                                                                                \
    }
    if (cfg != 0 && cfg != 4) throw Error(ERR_ARG, "launch_gemm_bf16x3: tile config 0 or 4");
    KV_BF_CASE(0, 0)
    KV_BF_CASE(0, 1)
    KV_BF_CASE(0, 2)
    KV_BF_CASE(1, 0)
    KV_BF_CASE(1, 1)
    KV_BF_CASE(1, 2)
    KV_BF_CASE(2, 0)
    KV_BF_CASE(2, 1)
    KV_BF_CASE(2, 2)
#undef KV_BF_CASE
    throw Error(ERR_ARG, "launch_gemm_bf16x3: bad op codes");
}

// ------------------------------------------------------------------------------------
// MPO fold
// ------------------------------------------------------------------------------------
// One workgroup column per task (an output (s', w') row of a block, P x Q elements), the
// task's P x Q elements spread over all threads of gridDim.y workgroups in row-major order
// (consecutive lanes on consecutive q, so every lane works even when Q < 256); the terms
// are summed in order, four loads issued together.
template <class T2>
__global__ __launch_bounds__(256) void wfold_kernel(const T2* __restrict__ in,
                                                    T2* __restrict__ out,
                                                    const WTask* __restrict__ tasks,
                                                    const WTerm* __restrict__ terms,
                                                    const int* __restrict__ stop, Mark* mark) {
    if (stop && *stop) return;
    write_mark(mark);
    using T = typename ScalarOf<T2>::T;
    const WTask tk = tasks[blockIdx.x];
    const WTerm* __restrict__ tt = terms + tk.term_begin;
    const int nt = tk.term_count, Q = tk.Q;
    const int PQ = tk.P * Q;
    if constexpr (sizeof(T2) == 8) {
        // FP32 complex: two neighbouring q per thread as one 16-byte load per term, when every
        // offset and stride of the task is even (the addresses are then 16-byte aligned)
        int64_t odd = tk.out_base | tk.out_pstride | (int64_t)Q;
        for (int t = 0; t < nt; ++t) odd |= tt[t].in_base | tt[t].in_pstride;
        if ((odd & 1) == 0) {
            const int Q2 = Q >> 1, PQ2 = PQ >> 1;
            for (int e = blockIdx.y * 256 + threadIdx.x; e < PQ2; e += gridDim.y * 256) {
                const int p = e / Q2, q = 2 * (e - p * Q2);
                float re0 = 0.f, im0 = 0.f, re1 = 0.f, im1 = 0.f;
#pragma unroll 4
                for (int t = 0; t < nt; ++t) {
                    const WTerm w = tt[t];
                    const float4 v = *reinterpret_cast<const float4*>(in + w.in_base + (int64_t)p * w.in_pstride + q);
                    const float wr = (float)w.re, wi = (float)w.im;
                    re0 += wr * v.x - wi * v.y;
                    im0 += wr * v.y + wi * v.x;
                    re1 += wr * v.z - wi * v.w;
                    im1 += wr * v.w + wi * v.z;
                }
                *reinterpret_cast<float4*>(out + tk.out_base + (int64_t)p * tk.out_pstride + q) =
                    make_float4(re0, im0, re1, im1);
            }
            return;
        }
    }
    for (int e = blockIdx.y * 256 + threadIdx.x; e < PQ; e += gridDim.y * 256) {
        const int p = e / Q, q = e - p * Q;
        T re = 0, im = 0;
        int t = 0;
        for (; t + 4 <= nt; t += 4) {
            T2 v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = in[tt[t + u].in_base + (int64_t)p * tt[t + u].in_pstride + q];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const T wr = (T)tt[t + u].re, wi = (T)tt[t + u].im;
                re += wr * v[u].x - wi * v[u].y;
                im += wr * v[u].y + wi * v[u].x;
            }
        }
        for (; t < nt; ++t) {
            const WTerm w = tt[t];
            const T2 v = in[w.in_base + (int64_t)p * w.in_pstride + q];
            const T wr = (T)w.re, wi = (T)w.im;
            re += wr * v.x - wi * v.y;
            im += wr * v.y + wi * v.x;
        }
        T2 o;
        o.x = re;
        o.y = im;
        out[tk.out_base + (int64_t)p * tk.out_pstride + q] = o;
    }
}

template <class T2>
void launch_wfold(hipStream_t st, const T2* in, T2* out, const WTask* tasks, int ntasks,
                  const WTerm* terms, int64_t maxPQ, const int* stop, Mark* mark) {
    if (ntasks <= 0) return;
    int64_t gy = (maxPQ + 255) / 256;
    if (gy > 64) gy = 64;
    if (gy < 1) gy = 1;
    hipLaunchKernelGGL((wfold_kernel<T2>), dim3(ntasks, (unsigned)gy), dim3(256), 0, st, in, out, tasks, terms, stop,
                       mark);
    KV_HIP(hipGetLastError());
}
template void launch_wfold<double2>(hipStream_t, const double2*, double2*, const WTask*, int,
                                    const WTerm*, int64_t, const int*, Mark*);
template void launch_wfold<float2>(hipStream_t, const float2*, float2*, const WTask*, int,
                                   const WTerm*, int64_t, const int*, Mark*);

__global__ __launch_bounds__(64) void wcompose_kernel(const WComposeTask* __restrict__ tasks2,
                                                      const WComposeTerm* __restrict__ terms2,
                                                      const WTask* __restrict__ tasks1,
                                                      const WTerm* __restrict__ terms1, WTask* __restrict__ tasks,
                                                      WTerm* __restrict__ terms) {
    const WComposeTask c = tasks2[blockIdx.x];
    for (int s1 = threadIdx.x; s1 < c.S1; s1 += 64) wcompose_expand(c, s1, terms2, tasks1, terms1, tasks, terms);
}

void launch_wcompose(hipStream_t st, const WComposeTask* tasks2, int n2, const WComposeTerm* terms2,
                     const WTask* tasks1, const WTerm* terms1, WTask* tasks, WTerm* terms) {
    if (n2 <= 0) return;
    hipLaunchKernelGGL(wcompose_kernel, dim3(n2), dim3(64), 0, st, tasks2, terms2, tasks1, terms1, tasks, terms);
    KV_HIP(hipGetLastError());
}

// ------------------------------------------------------------------------------------
// block permutation
// ------------------------------------------------------------------------------------
template <class T2>
__global__ __launch_bounds__(256) void perm_kernel(const T2* __restrict__ in,
                                                   T2* __restrict__ out,
                                                   const PermTask* __restrict__ tasks) {
    // fields are read through the pointer: a by-value copy indexed by r would live in
    // scratch memory
    const PermTask* tk = tasks + blockIdx.x;
    const int64_t size = tk->size, in_off = tk->in_off, out_off = tk->out_off;
    const int rank = tk->rank;
    for (int64_t e = (int64_t)blockIdx.y * blockDim.x + threadIdx.x; e < size;
         e += (int64_t)gridDim.y * blockDim.x) {
        int64_t rem = e, src = 0;
        for (int r = rank - 1; r >= 0; --r) {
            const int64_t sh = tk->oshape[r];
            const int64_t idx = rem % sh;
            rem /= sh;
            src += idx * tk->istride[r];
        }
        out[out_off + e] = in[in_off + src];
    }
}

template <class T2>
void launch_perm(hipStream_t st, const T2* in, T2* out, const PermTask* tasks, int ntasks,
                 int64_t maxsize) {
    if (ntasks <= 0 || maxsize <= 0) return;
    int64_t gy = (maxsize + 255) / 256;
    if (gy > 1024) gy = 1024;
    hipLaunchKernelGGL((perm_kernel<T2>), dim3(ntasks, (unsigned)gy), dim3(256), 0, st, in,
                       out, tasks);
    KV_HIP(hipGetLastError());
}
template void launch_perm<double2>(hipStream_t, const double2*, double2*, const PermTask*, int,
                                   int64_t);
template void launch_perm<float2>(hipStream_t, const float2*, float2*, const PermTask*, int,
                                  int64_t);

// ------------------------------------------------------------------------------------
// 2-D strided copies with optional diagonal scaling
// ------------------------------------------------------------------------------------
template <class T2>
__global__ __launch_bounds__(256) void copy2d_kernel(const T2* __restrict__ src,
                                                     T2* __restrict__ dst,
                                                     const Copy2D* __restrict__ cps,
                                                     const double* __restrict__ scale) {
    using T = typename ScalarOf<T2>::T;
    const Copy2D c = cps[blockIdx.x];
    for (int r = blockIdx.y; r < c.rows; r += gridDim.y) {
        for (int q = threadIdx.x; q < c.cols; q += blockDim.x) {
            T2 v = src[c.src_off + (int64_t)r * c.src_ld + q];
            if (c.scale_mode == 1) {
                const T f = (T)scale[c.scale_off + r];
                v.x *= f;
                v.y *= f;
            } else if (c.scale_mode == 2) {
                const T f = (T)scale[c.scale_off + q];
                v.x *= f;
                v.y *= f;
            }
            dst[c.dst_off + (int64_t)r * c.dst_ld + q] = v;
        }
    }
}

template <class T2>
void launch_copy2d(hipStream_t st, const T2* src, T2* dst, const Copy2D* cps, int ncopies,
                   int maxrows, const double* scale) {
    if (ncopies <= 0 || maxrows <= 0) return;
    const int gy = maxrows < 256 ? maxrows : 256;
    hipLaunchKernelGGL((copy2d_kernel<T2>), dim3(ncopies, gy), dim3(256), 0, st, src, dst, cps,
                       scale);
    KV_HIP(hipGetLastError());
}
template void launch_copy2d<double2>(hipStream_t, const double2*, double2*, const Copy2D*, int,
                                     int, const double*);

// dst[c*ld_dst + r] = conj(src[r*ld_src + c]) for r < rows, c < cols (32x32 LDS tiles)
__global__ __launch_bounds__(256) void ctranspose_kernel(const double2* __restrict__ src,
                                                         double2* __restrict__ dst, int rows,
                                                         int cols, int ld_src, int ld_dst) {
    __shared__ double2 t[32][33];
    const int r0 = blockIdx.y * 32, c0 = blockIdx.x * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int i = ty; i < 32; i += 8) {
        const int r = r0 + i, c = c0 + tx;
        if (r < rows && c < cols) t[i][tx] = src[(int64_t)r * ld_src + c];
    }
    __syncthreads();
    for (int i = ty; i < 32; i += 8) {
        const int c = c0 + i, r = r0 + tx;
        if (r < rows && c < cols) {
            const double2 v = t[tx][i];
            dst[(int64_t)c * ld_dst + r] = make_double2(v.x, -v.y);
        }
    }
}

void launch_ctranspose(hipStream_t st, const double2* src, double2* dst, int rows, int cols,
                       int ld_src, int ld_dst) {
    if (rows <= 0 || cols <= 0) return;
    hipLaunchKernelGGL(ctranspose_kernel, dim3((cols + 31) / 32, (rows + 31) / 32), dim3(256), 0,
                       st, src, dst, rows, cols, ld_src, ld_dst);
    KV_HIP(hipGetLastError());
}

// ------------------------------------------------------------------------------------
// FP64 vector algebra
// ------------------------------------------------------------------------------------
constexpr int RED_BLOCKS = kRedBlocks;

__global__ __launch_bounds__(256) void zero_kernel(uint32_t* __restrict__ p, int64_t n) {
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256)
        p[e] = 0u;
}

// Zero fill by a kernel (not hipMemsetAsync), so the call stays safe inside captured graphs.
void launch_zero(hipStream_t st, void* p, size_t bytes) {
    if (!bytes) return;
    const int64_t n = (int64_t)(bytes / 4);
    int64_t b = (n + 255) / 256;
    if (b > 4096) b = 4096;
    if (b < 1) b = 1;
    hipLaunchKernelGGL(zero_kernel, dim3((unsigned)b), dim3(256), 0, st, (uint32_t*)p, n);
    KV_HIP(hipGetLastError());
}

__global__ __launch_bounds__(256) void dotc_partial_kernel(const double2* __restrict__ a,
                                                           const double2* __restrict__ b,
                                                           int64_t n, double* __restrict__ part) {
    __shared__ double sr[256], si[256];
    double re = 0, im = 0;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
        const double2 x = a[e], y = b[e];
        re += x.x * y.x + x.y * y.y;  // conj(x) * y
        im += x.x * y.y - x.y * y.x;
    }
    sr[threadIdx.x] = re;
    si[threadIdx.x] = im;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            sr[threadIdx.x] += sr[threadIdx.x + s];
            si[threadIdx.x] += si[threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = sr[0];
        part[2 * blockIdx.x + 1] = si[0];
    }
}

__global__ __launch_bounds__(256) void reduce2_final_kernel(const double* __restrict__ part,
                                                            int nb, double* __restrict__ out,
                                                            int ncomp) {
    __shared__ double s0[256], s1[256];
    double a = 0, b = 0;
    for (int i = threadIdx.x; i < nb; i += 256) {
        a += part[ncomp * i];
        if (ncomp == 2) b += part[ncomp * i + 1];
    }
    s0[threadIdx.x] = a;
    s1[threadIdx.x] = b;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            s0[threadIdx.x] += s0[threadIdx.x + s];
            s1[threadIdx.x] += s1[threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        out[0] = s0[0];
        if (ncomp == 2) out[1] = s1[0];
    }
}

static int red_blocks(int64_t n) {
    int64_t b = (n + 255) / 256;
    if (b > RED_BLOCKS) b = RED_BLOCKS;
    if (b < 1) b = 1;
    return (int)b;
}

void launch_dotc(hipStream_t st, const double2* a, const double2* b, int64_t n, double2* out,
                 double* scratch) {
    const int nb = red_blocks(n);
    hipLaunchKernelGGL(dotc_partial_kernel, dim3(nb), dim3(256), 0, st, a, b, n, scratch);
    KV_HIP(hipGetLastError());
    hipLaunchKernelGGL(reduce2_final_kernel, dim3(1), dim3(256), 0, st, scratch, nb,
                       reinterpret_cast<double*>(out), 2);
    KV_HIP(hipGetLastError());
}

__global__ __launch_bounds__(256) void nrm2sq_partial_kernel(const double2* __restrict__ a,
                                                             int64_t n, double* __restrict__ part) {
    __shared__ double sr[256];
    double re = 0;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
        const double2 x = a[e];
        re += x.x * x.x + x.y * x.y;
    }
    sr[threadIdx.x] = re;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) sr[threadIdx.x] += sr[threadIdx.x + s];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sr[0];
}

void launch_nrm2sq(hipStream_t st, const double2* a, int64_t n, double* out, double* scratch) {
    const int nb = red_blocks(n);
    hipLaunchKernelGGL(nrm2sq_partial_kernel, dim3(nb), dim3(256), 0, st, a, n, scratch);
    KV_HIP(hipGetLastError());
    hipLaunchKernelGGL(reduce2_final_kernel, dim3(1), dim3(256), 0, st, scratch, nb, out, 1);
    KV_HIP(hipGetLastError());
}

static unsigned ew_blocks(int64_t n) {
    int64_t b = (n + 255) / 256;
    if (b > 4096) b = 4096;
    if (b < 1) b = 1;
    return (unsigned)b;
}

// ---- Lanczos recurrence -------------------------------------------------------------
// One iteration after h = H v_k: beta = <h|v_{k-1}>, h -= beta v_{k-1}, alpha = <h|v_k>,
// h -= alpha v_k, |h|^2, v_{k+1} = h / |h|, in the reference's order and with one reduction
// tree throughout: 256-element chunks dealt round-robin to up to RED_BLOCKS workgroups, a
// pairwise tree over a workgroup's 256 lanes, then the same tree over the workgroups.
// Long vectors (bound by HBM, 11 passes per iteration) take one launch per phase, each
// forming the total of the phase before from its partials (at most 16 KB from L2) instead of
// waiting for a one-workgroup kernel; short ones (kLanczosSmall: bound by launches, 2.2 us and
// a gap each) run the whole recurrence in one workgroup with h in registers.  The launches
// of an iteration read its stop word first, so the host may queue the next iteration before
// it has seen the scalars of this one.
// One site at D = 16, 4 levels (nine iterations of 11 launches, a copy and a wait each): 796 us a
// call before, 337 now; the middle bond at D = 256, 16 levels with its SVD 32.0 -> 29.3 ms.

// Total of nb partials (NC interleaved components), formed by every wave of a 256-thread
// workgroup; sh holds 256 values per component.
template <int NC>
__device__ inline double2 partials_total(const double* __restrict__ part, int nb, double (*sh)[256]) {
    double a = 0, b = 0;
    for (int i = threadIdx.x; i < nb; i += 256) {
        a += part[NC * i];
        if (NC == 2) b += part[NC * i + 1];
    }
    __syncthreads();
    sh[0][threadIdx.x] = a;
    if (NC == 2) sh[1][threadIdx.x] = b;
    __syncthreads();
    const int t = threadIdx.x & 63;
    double2 r = make_double2(0, 0);
    r.x = lane_first(tree64((sh[0][t] + sh[0][t + 128]) + (sh[0][t + 64] + sh[0][t + 192])));
    if (NC == 2) r.y = lane_first(tree64((sh[1][t] + sh[1][t + 128]) + (sh[1][t + 64] + sh[1][t + 192])));
    return r;
}

// A workgroup's partial from its 256 lanes' sums.
template <int NC>
__device__ inline void partial_store(double a, double b, double* __restrict__ part, double (*sh)[256]) {
    __syncthreads();
    sh[0][threadIdx.x] = a;
    if (NC == 2) sh[1][threadIdx.x] = b;
    __syncthreads();
    if (threadIdx.x >= 64) return;
    const int t = threadIdx.x;
    const double x = tree64((sh[0][t] + sh[0][t + 128]) + (sh[0][t + 64] + sh[0][t + 192]));
    double y = 0;
    if (NC == 2) y = tree64((sh[1][t] + sh[1][t + 128]) + (sh[1][t + 64] + sh[1][t + 192]));
    if (t == 0) {
        part[NC * blockIdx.x] = x;
        if (NC == 2) part[NC * blockIdx.x + 1] = y;
    }
}

// What the host reads of iteration k; `seen` is written last.
__device__ inline void lanczos_publish(LanczosHost* rec, double2 beta, double2 alpha, double nsq, double err,
                                       unsigned long long tag) {
    // stores past the caches, and a wait for them in place of a system-scope fence, which would
    // write back the whole L2
    auto put = [](double* p, double v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM); };
    put(&rec->beta_re, beta.x);
    put(&rec->beta_im, beta.y);
    put(&rec->alpha_re, alpha.x);
    put(&rec->alpha_im, alpha.y);
    put(&rec->nsq, nsq);
    put(&rec->err, err);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __hip_atomic_store(&rec->seen, tag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// partial sums of |x|^2; clears the call's stop words and sets err[0] = 1.
__global__ __launch_bounds__(256) void lanczos_begin_kernel(const double2* __restrict__ x, int64_t n,
                                                            double* __restrict__ part, LanczosDev* __restrict__ st) {
    __shared__ double sh[1][256];
    if (blockIdx.x == 0 && threadIdx.x <= kLanczosMax) {
        st->stop[threadIdx.x] = 0;
        if (threadIdx.x == 0) st->err[0] = 1.0;
    }
    double re = 0;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
        const double2 v = x[e];
        re += v.x * v.x + v.y * v.y;
    }
    partial_store<1>(re, 0, part, sh);
}

// v_0 = x / |x| from the partials of lanczos_begin_kernel.
__global__ __launch_bounds__(256) void lanczos_first_kernel(const double2* __restrict__ x, double2* __restrict__ v0,
                                                            int64_t n, const double* __restrict__ part, int nb) {
    __shared__ double sh[1][256];
    const double f = 1.0 / sqrt(partials_total<1>(part, nb, sh).x);
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
        double2 v = x[e];
        v.x *= f;
        v.y *= f;
        v0[e] = v;
    }
}

// Phases of one iteration.  DOT: partials of <h|z> alone (the first phase).  SUBDOT: c = the
// total of the phase before, kept in *c_out; h -= c x; partials of <h|z>.  SUBNRM: the same with
// |h|^2.
enum { LZ_DOT, LZ_SUBDOT, LZ_SUBNRM };
template <int PHASE>
__global__ __launch_bounds__(256) void lanczos_phase_kernel(double2* __restrict__ h, const double2* __restrict__ x,
                                                            const double2* __restrict__ z, int64_t n,
                                                            const double* __restrict__ in, int nb,
                                                            double* __restrict__ out, double2* __restrict__ c_out,
                                                            const int* __restrict__ stop, Mark* mark) {
    if (*stop) return;
    write_mark(mark);
    __shared__ double sh[2][256];
    double2 c = make_double2(0, 0);
    if constexpr (PHASE != LZ_DOT) {
        c = partials_total<2>(in, nb, sh);
        if (blockIdx.x == 0 && threadIdx.x == 0) *c_out = c;
    }
    double re = 0, im = 0;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
        double2 o = h[e];
        if constexpr (PHASE != LZ_DOT) {
            const double2 v = x[e];
            o.x -= c.x * v.x - c.y * v.y;
            o.y -= c.x * v.y + c.y * v.x;
            h[e] = o;
        }
        if constexpr (PHASE == LZ_SUBNRM) {
            re += o.x * o.x + o.y * o.y;
        } else {
            const double2 w = z[e];
            re += o.x * w.x + o.y * w.y;  // conj(o) * w
            im += o.x * w.y - o.y * w.x;
        }
    }
    partial_store<PHASE == LZ_SUBNRM ? 1 : 2>(re, im, out, sh);
}

// |h|^2 from its partials, err_{k+1} = err_k |h| and the stop word of iteration k + 1; unless
// stopped, v_{k+1} = h / |h|.
__global__ __launch_bounds__(256) void lanczos_next_kernel(const double2* __restrict__ h, double2* __restrict__ vn,
                                                           int64_t n, const double* __restrict__ part, int nb,
                                                           LanczosDev* __restrict__ st, int k, double tol,
                                                           LanczosHost* rec, unsigned long long tag) {
    if (st->stop[k]) return;
    __shared__ double sh[1][256];
    const double nsq = partials_total<1>(part, nb, sh).x;
    const double err = st->err[k] * sqrt(nsq);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        st->err[k + 1] = err;
        st->stop[k + 1] = !(err > tol);
        lanczos_publish(rec, st->beta, st->alpha, nsq, err, tag);
    }
    if (!(err > tol)) return;
    const double f = 1.0 / sqrt(nsq);
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
        double2 v = h[e];
        v.x *= f;
        v.y *= f;
        vn[e] = v;
    }
}

// One wave's partial of a 256-element chunk: lane t holds elements t, t + 64, t + 128, t + 192.
__device__ inline double chunk_sum(const double (&p)[4]) { return tree64((p[0] + p[2]) + (p[1] + p[3])); }
// Total of nb <= 64 chunk partials, in every lane.
__device__ inline double chunks_total(const double* sh, int nb) {
    const int t = threadIdx.x & 63;
    return lane_first(tree64(t < nb ? sh[t] : 0.0));
}

// v_0 = x / |x| and the call's state, in one workgroup (n <= kLanczosSmall).
__global__ __launch_bounds__(1024) void lanczos_first_small_kernel(const double2* __restrict__ x,
                                                                   double2* __restrict__ v0, int n,
                                                                   LanczosDev* __restrict__ st) {
    __shared__ double sh[64];
    const int wave = threadIdx.x >> 6, t = threadIdx.x & 63;
    const int nb = (n + 255) / 256;
    if (threadIdx.x <= kLanczosMax) {
        st->stop[threadIdx.x] = 0;
        if (threadIdx.x == 0) st->err[0] = 1.0;
    }
    for (int b = wave; b < nb; b += 16) {
        double p[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int e = b * 256 + j * 64 + t;
            const double2 v = e < n ? x[e] : make_double2(0, 0);
            p[j] = v.x * v.x + v.y * v.y;
        }
        const double s = chunk_sum(p);
        if (t == 0) sh[b] = s;
    }
    __syncthreads();
    const double f = 1.0 / sqrt(chunks_total(sh, nb));
    for (int e = threadIdx.x; e < n; e += 1024) {
        double2 v = x[e];
        v.x *= f;
        v.y *= f;
        v0[e] = v;
    }
}

// The whole recurrence of one iteration in one workgroup (n <= kLanczosSmall = 16 waves x NC
// chunks x 256): h stays in registers from its first read to v_{k+1}.
template <int NC>
__global__ __launch_bounds__(1024) void lanczos_small_kernel(const double2* __restrict__ h,
                                                             const double2* __restrict__ vkm,
                                                             const double2* __restrict__ vk,
                                                             double2* __restrict__ vn, int n,
                                                             LanczosDev* __restrict__ st, int k, double tol,
                                                             LanczosHost* rec, unsigned long long tag, Mark* mark) {
    if (st->stop[k]) return;
    write_mark(mark);
    __shared__ double sr[64], si[64];
    const int wave = threadIdx.x >> 6, t = threadIdx.x & 63;
    const int nb = (n + 255) / 256;
    // v_{k-1}, then v_k: kept beside h where the registers hold both (128 per lane), else read
    // twice (from L2)
    constexpr bool KEEP = NC <= 2;
    double2 r[NC][4], v[KEEP ? NC : 1][4];
    auto at = [&](const double2* p, int c, int j) -> double2 {
        const int e = (wave + 16 * c) * 256 + j * 64 + t;
        return e < n ? p[e] : make_double2(0, 0);
    };
    const double2* src = k > 0 ? vkm : vk;
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            r[c][j] = at(h, c, j);
            if (KEEP) v[c][j] = at(src, c, j);
        }
    auto dot = [&]() -> double2 {  // <r|v>
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            double p[4], q[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const double2 w = KEEP ? v[KEEP ? c : 0][j] : at(src, c, j);
                p[j] = r[c][j].x * w.x + r[c][j].y * w.y;
                q[j] = r[c][j].x * w.y - r[c][j].y * w.x;
            }
            const double a = chunk_sum(p), b = chunk_sum(q);
            if (t == 0) {
                sr[wave + 16 * c] = a;
                si[wave + 16 * c] = b;
            }
        }
        __syncthreads();
        const double2 d = make_double2(chunks_total(sr, nb), chunks_total(si, nb));
        __syncthreads();
        return d;
    };
    auto sub = [&](double2 d) {  // r -= d v
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const double2 w = KEEP ? v[KEEP ? c : 0][j] : at(src, c, j);
                r[c][j].x -= d.x * w.x - d.y * w.y;
                r[c][j].y -= d.x * w.y + d.y * w.x;
            }
    };
    double2 beta = make_double2(0, 0);
    if (k > 0) {
        beta = dot();
        sub(beta);
        src = vk;
        if (KEEP) {
#pragma unroll
            for (int c = 0; c < NC; ++c)
#pragma unroll
                for (int j = 0; j < 4; ++j) v[KEEP ? c : 0][j] = at(src, c, j);
        }
    }
    const double2 alpha = dot();
    sub(alpha);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        double p[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) p[j] = r[c][j].x * r[c][j].x + r[c][j].y * r[c][j].y;
        const double a = chunk_sum(p);
        if (t == 0) sr[wave + 16 * c] = a;
    }
    __syncthreads();
    const double nsq = chunks_total(sr, nb);
    const double err = st->err[k] * sqrt(nsq);
    if (threadIdx.x == 0) {
        st->err[k + 1] = err;
        st->stop[k + 1] = !(err > tol);
        lanczos_publish(rec, beta, alpha, nsq, err, tag);
    }
    if (!(err > tol)) return;
    const double f = 1.0 / sqrt(nsq);
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int e = (wave + 16 * c) * 256 + j * 64 + t;
            if (e < n) vn[e] = make_double2(f * r[c][j].x, f * r[c][j].y);
        }
}

// out = sum_i c_i V_i and the partials of |out|^2; the coefficients travel as an argument.
struct LincombArgs {
    double2 c[kLanczosMax];
};
__global__ __launch_bounds__(256) void lincomb_kernel(double2* __restrict__ out, const double2* __restrict__ V,
                                                      LincombArgs a, int nv, int64_t n, double* __restrict__ part) {
    __shared__ double sh[1][256];
    double sq = 0;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
        double re = 0, im = 0;
        for (int i = 0; i < nv; ++i) {
            const double2 v = V[(int64_t)i * n + e];
            const double2 ci = a.c[i];
            re += ci.x * v.x - ci.y * v.y;
            im += ci.x * v.y + ci.y * v.x;
        }
        out[e] = make_double2(re, im);
        sq += re * re + im * im;
    }
    partial_store<1>(sq, 0, part, sh);
}

// The total of nb partials to the host.
__global__ __launch_bounds__(256) void lanczos_end_kernel(const double* __restrict__ part, int nb, LanczosHost* rec,
                                                          unsigned long long tag) {
    __shared__ double sh[1][256];
    const double s = partials_total<1>(part, nb, sh).x;
    if (threadIdx.x == 0) lanczos_publish(rec, make_double2(0, 0), make_double2(0, 0), s, 0, tag);
}

void launch_lanczos_begin(hipStream_t st, const double2* x, double2* v0, int64_t n, double* part, LanczosDev* dev) {
    if (n <= kLanczosSmall) {
        hipLaunchKernelGGL(lanczos_first_small_kernel, dim3(1), dim3(1024), 0, st, x, v0, (int)n, dev);
        KV_HIP(hipGetLastError());
        return;
    }
    const int nb = red_blocks(n);
    hipLaunchKernelGGL(lanczos_begin_kernel, dim3(nb), dim3(256), 0, st, x, n, part, dev);
    KV_HIP(hipGetLastError());
    hipLaunchKernelGGL(lanczos_first_kernel, dim3(nb), dim3(256), 0, st, x, v0, n, part, nb);
    KV_HIP(hipGetLastError());
}

void launch_lanczos_step(hipStream_t st, double2* h, const double2* vkm, const double2* vk, double2* vn, int64_t n,
                         double* part, LanczosDev* dev, int k, double tol, LanczosHost* rec, uint64_t tag, Mark* mark) {
    if (n <= kLanczosSmall) {
        static_assert(kLanczosSmall == 3 * 16 * 256, "the chunks of the largest variant");
        const auto f = n <= kLanczosSmall / 3       ? lanczos_small_kernel<1>
                       : n <= 2 * kLanczosSmall / 3 ? lanczos_small_kernel<2>
                                                    : lanczos_small_kernel<3>;
        hipLaunchKernelGGL(f, dim3(1), dim3(1024), 0, st, h, vkm, vk, vn, (int)n, dev, k, tol, rec,
                           (unsigned long long)tag, mark);
        KV_HIP(hipGetLastError());
        return;
    }
    const int nb = red_blocks(n);
    const dim3 grid(nb), block(256);
    double *pa = part, *pb = part + 2 * RED_BLOCKS, *pc = part + 4 * RED_BLOCKS;
    const int* stop = &dev->stop[k];
    if (k > 0) {
        hipLaunchKernelGGL(lanczos_phase_kernel<LZ_DOT>, grid, block, 0, st, h, nullptr, vkm, n, nullptr, 0, pa,
                           nullptr, stop, mark);
        KV_HIP(hipGetLastError());
        hipLaunchKernelGGL(lanczos_phase_kernel<LZ_SUBDOT>, grid, block, 0, st, h, vkm, vk, n, pa, nb, pb, &dev->beta,
                           stop, nullptr);
    } else {
        hipLaunchKernelGGL(lanczos_phase_kernel<LZ_DOT>, grid, block, 0, st, h, nullptr, vk, n, nullptr, 0, pb,
                           nullptr, stop, mark);
    }
    KV_HIP(hipGetLastError());
    hipLaunchKernelGGL(lanczos_phase_kernel<LZ_SUBNRM>, grid, block, 0, st, h, vk, nullptr, n, pb, nb, pc, &dev->alpha,
                       stop, nullptr);
    KV_HIP(hipGetLastError());
    hipLaunchKernelGGL(lanczos_next_kernel, grid, block, 0, st, h, vn, n, pc, nb, dev, k, tol, rec,
                       (unsigned long long)tag);
    KV_HIP(hipGetLastError());
}

void launch_lanczos_end(hipStream_t st, double2* out, const double2* V, const double2* c, int nv, int64_t n,
                        double* part, LanczosHost* rec, uint64_t tag) {
    const int nb = red_blocks(n);
    LincombArgs a{};
    for (int i = 0; i < nv; ++i) a.c[i] = c[i];
    hipLaunchKernelGGL(lincomb_kernel, dim3(nb), dim3(256), 0, st, out, V, a, nv, n, part);
    KV_HIP(hipGetLastError());
    hipLaunchKernelGGL(lanczos_end_kernel, dim3(1), dim3(256), 0, st, part, nb, rec, (unsigned long long)tag);
    KV_HIP(hipGetLastError());
}

__global__ __launch_bounds__(256) void scale_kernel(double2* __restrict__ dst,
                                                    const double2* __restrict__ src, double s,
                                                    int64_t n) {
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
        double2 v = src[e];
        v.x *= s;
        v.y *= s;
        dst[e] = v;
    }
}

void launch_scale(hipStream_t st, double2* dst, const double2* src, double s, int64_t n) {
    if (n <= 0) return;
    hipLaunchKernelGGL(scale_kernel, dim3(ew_blocks(n)), dim3(256), 0, st, dst, src, s, n);
    KV_HIP(hipGetLastError());
}

// out = a*x + b*y elementwise (complex a, b); x or y may be null (term dropped).
__global__ __launch_bounds__(256) void zaxpby_kernel(double2* __restrict__ out,
                                                     const double2* __restrict__ x,
                                                     const double2* __restrict__ y, double2 a,
                                                     double2 b, int64_t n) {
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
        double re = 0, im = 0;
        if (x) {
            const double2 v = x[e];
            re += a.x * v.x - a.y * v.y;
            im += a.x * v.y + a.y * v.x;
        }
        if (y) {
            const double2 v = y[e];
            re += b.x * v.x - b.y * v.y;
            im += b.x * v.y + b.y * v.x;
        }
        out[e] = make_double2(re, im);
    }
}

void launch_zaxpby(hipStream_t st, double2* out, const double2* x, const double2* y, double2 a,
                   double2 b, int64_t n) {
    if (n <= 0) return;
    hipLaunchKernelGGL(zaxpby_kernel, dim3(ew_blocks(n)), dim3(256), 0, st, out, x, y, a, b, n);
    KV_HIP(hipGetLastError());
}

__global__ __launch_bounds__(256) void f64_to_f32_kernel(const double2* __restrict__ s,
                                                         float2* __restrict__ d, int64_t n,
                                                         const int* __restrict__ stop) {
    if (stop && *stop) return;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
        const double2 v = s[e];
        d[e] = make_float2((float)v.x, (float)v.y);
    }
}

void launch_f64_to_f32(hipStream_t st, const double2* src, float2* dst, int64_t n, const int* stop) {
    if (n <= 0) return;
    hipLaunchKernelGGL(f64_to_f32_kernel, dim3(ew_blocks(n)), dim3(256), 0, st, src, dst, n, stop);
    KV_HIP(hipGetLastError());
}

__global__ __launch_bounds__(256) void f32_to_f64_kernel(const float2* __restrict__ s,
                                                         double2* __restrict__ d, double f,
                                                         int64_t n, const int* __restrict__ stop, Mark* mark) {
    if (stop && *stop) return;
    write_mark(mark);
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
        const float2 v = s[e];
        d[e] = make_double2(f * (double)v.x, f * (double)v.y);
    }
}

void launch_f32_to_f64(hipStream_t st, const float2* src, double2* dst, double s, int64_t n, const int* stop,
                       Mark* mark) {
    if (n <= 0) return;
    hipLaunchKernelGGL(f32_to_f64_kernel, dim3(ew_blocks(n)), dim3(256), 0, st, src, dst, s, n, stop, mark);
    KV_HIP(hipGetLastError());
}

// ---- SVD of small sectors ------------------------------------------------------------------
// One workgroup per matrix whose smaller side n is at most kJacobiMax, all sectors of a bond in
// one launch.  The tall form A (m x n: M, or M^H where M is wide) is reduced by Householder
// reflections (LAPACK zgeqrf's formulas) to R, one-sided Jacobi rotations W orthogonalise the
// columns of R^H in LDS (R^H W = Y, Y_i = s_i x_i; Drmac and Veselic, SIAM J. Matrix Anal. Appl.
// 29 (2008): the triangular factor's columns are nearly orthogonal already, and relative
// accuracy of small singular values survives), and the reflectors carry W back: A = (Q W) S X^H.
// Both factors are orthonormal to rounding whatever the spectrum.
// Bound by latency: one barrier per reflector and per rotation round.  A wave takes a column, its
// rows strided over the lanes so that a lane rereads only what it wrote; the wave that updates
// the next pivot column forms its reflector in the same step.  A half wave takes a pair of
// columns (n / 2 disjoint pairs a round).
// A bond of two 768 x 32 sectors: 0.52 ms (reduction 0.33, rotations 0.16), 3.7 through zgesvdj.
constexpr double kJacobiTol = 4e-16;  // x sqrt(n): |x_i^H x_j| against |x_i| |x_j|
constexpr int kJacobiSweeps = 40;
// Squared norm, next to a largest entry of about one, below which a column counts as zero.  The
// columns of a rank-deficient factor that can be orthogonal to nothing lose sixteen digits of
// length with every sweep and would be rotated until they underflow.
constexpr double kJacobiZero = 1e-60;

__device__ inline double wave_all(double v) { return lane_first(tree64(v)); }
// the sum over each half wave in all of its lanes
__device__ inline double half_all(double v) {
    v = row_all(v);
    return v + __shfl_xor(v, 16);
}

// a column's rows lane, lane + 64, ...: in registers (NT > 0, m <= 64 NT) or in memory
template <int NT>
struct ColView {
    double2 r[NT ? NT : 1];
    double2* p;
    int m, nt, lane;
    __device__ ColView(double2* q, int m_, int lane_) : p(q), m(m_), nt((m_ + 63) >> 6), lane(lane_) {}
    __device__ void load() {
        if constexpr (NT > 0) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int i = lane + 64 * t;
                r[t] = i < m ? p[i] : make_double2(0, 0);
            }
        }
    }
    // f(i, value) for this lane's rows i >= lo; store: the value is written back
    template <class F>
    __device__ void each(int lo, bool store, F f) {
        if constexpr (NT > 0) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int i = lane + 64 * t;
                if (i >= lo && i < m) {
                    f(i, r[t]);
                    if (store) p[i] = r[t];
                }
            }
        } else {
            for (int i = lane + (lo & ~63); i < m; i += 64) {
                if (i < lo) continue;
                double2 v = p[i];
                f(i, v);
                if (store) p[i] = v;
            }
        }
    }
};

template <int NT, int THREADS>
__global__ __launch_bounds__(THREADS) void jacobi_svd_kernel(const SvdJob* __restrict__ jobs) {
    constexpr int NW = THREADS / 64;
    extern __shared__ double2 lds[];  // X (n x n), W (n x n)
    __shared__ double red[NW];
    __shared__ double2 tau[kJacobiMax];
    __shared__ double rdiag[kJacobiMax], nrm[kJacobiMax];
    __shared__ int ord[kJacobiMax], rotated;
    const SvdJob J = jobs[blockIdx.x];
    const bool tall = J.nr >= J.nc;
    const int n = tall ? J.nc : J.nr, m = tall ? J.nr : J.nc;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    double2* A = J.A;

    // the largest component sets a power-of-two scale, so that squares neither overflow nor
    // vanish next to the largest value
    double amax = 0;
    bool bad = false;
    for (int e = tid; e < m * n; e += THREADS) {
        const double2 v = J.M[e];
        const double a = fmax(fabs(v.x), fabs(v.y));
        bad = bad || !(fabs(v.x) <= 1.7976931348623157e308 && fabs(v.y) <= 1.7976931348623157e308);
        amax = fmax(amax, a);
    }
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) amax = fmax(amax, __shfl_xor(amax, s));
    if (lane == 0) red[wave] = amax;
    if (__syncthreads_or(bad)) {  // a NaN or an infinity: no decomposition
        if (tid < n) J.S[tid] = __longlong_as_double(0x7ff8000000000000ll);
        return;
    }
    amax = 0;
    for (int w = 0; w < NW; ++w) amax = fmax(amax, red[w]);
    // a sector that goes to zgesvd all the same (two of 1024 x 40, all zero: 9.8 ms with the
    // decomposition before it, 8.9 without)
    auto zero_end = [&] {
        if (tid < n) J.S[tid] = tid + 1 < n ? 1.0 : 0.0;
    };
    if (J.zero_ends && amax == 0) {  // uniform
        zero_end();
        return;
    }
    int ex = 0;
    if (amax > 0) (void)frexp(amax, &ex);
    for (int e = tid; e < m * n; e += THREADS) {
        const double2 v = J.M[e];
        if (tall)
            A[(int64_t)(e % n) * m + e / n] = make_double2(ldexp(v.x, -ex), ldexp(v.y, -ex));
        else
            A[e] = make_double2(ldexp(v.x, -ex), -ldexp(v.y, -ex));
    }
    __syncthreads();

    // Householder QR; the reflector of column j overwrites its rows j.. (unit entry stored)
    auto reflector = [&](ColView<NT>& c, int j) {
        double2 head = make_double2(0, 0);
        double tail = 0;
        c.each(j, false, [&](int i, double2& v) {
            if (i == j)
                head = v;
            else
                tail += v.x * v.x + v.y * v.y;
        });
        tail = wave_all(tail);
        const double ar = __shfl(head.x, j & 63), ai = __shfl(head.y, j & 63);
        double2 tj = make_double2(0, 0), inv = make_double2(0, 0);
        double beta = ar;
        const double sq = ar * ar + ai * ai + tail;
        if (sq < 1e-280) {  // nothing left at 1e-140 of the largest entry: a zero column
            beta = 0;
        } else if (tail != 0 || ai != 0) {
            beta = -copysign(sqrt(sq), ar);
            tj = make_double2((beta - ar) / beta, -ai / beta);
            const double dr = ar - beta, d = dr * dr + ai * ai;  // 1 / (alpha - beta)
            inv = make_double2(dr / d, -ai / d);
        }
        c.each(j, true, [&](int i, double2& v) {
            v = i == j ? make_double2(1, 0) : make_double2(v.x * inv.x - v.y * inv.y, v.x * inv.y + v.y * inv.x);
        });
        if (lane == 0) {
            tau[j] = tj;
            rdiag[j] = beta;
        }
    };
    // column -= f v (v^H column) over rows j.., f = conj(tau_j)
    auto reflect = [&](ColView<NT>& c, int j, double2 f) {
        const double2* v = A + (int64_t)j * m;
        double wr = 0, wi = 0;
        c.each(j, false, [&](int i, double2& a) {
            const double2 u = v[i];
            wr += u.x * a.x + u.y * a.y;
            wi += u.x * a.y - u.y * a.x;
        });
        wr = wave_all(wr);
        wi = wave_all(wi);
        const double gr = f.x * wr - f.y * wi, gi = f.x * wi + f.y * wr;
        c.each(j, true, [&](int i, double2& a) {
            const double2 u = v[i];
            a.x -= u.x * gr - u.y * gi;
            a.y -= u.x * gi + u.y * gr;
        });
    };
    if (wave == 0) {
        ColView<NT> c(A, m, lane);
        c.load();
        reflector(c, 0);
    }
    __syncthreads();
    for (int j = 0; j + 1 < n; ++j) {
        const double2 f = make_double2(tau[j].x, -tau[j].y);
        for (int k = j + 1 + wave; k < n; k += NW) {
            ColView<NT> c(A + (int64_t)k * m, m, lane);
            c.load();
            reflect(c, j, f);
            if (k == j + 1) reflector(c, j + 1);
        }
        __syncthreads();
    }

    if (J.zero_ends) {
        bool zero = false;
        for (int i = 0; i < n; ++i) zero = zero || rdiag[i] == 0;
        if (zero) {  // uniform
            zero_end();
            return;
        }
    }
    // X = R^H column by column, W = 1
    double2 *X = lds, *W = lds + n * n;
    for (int e = tid; e < n * n; e += THREADS) {
        const int i = e / n, r = e % n;
        double2 v = make_double2(0, 0);
        if (r > i) {
            v = A[(int64_t)r * m + i];
            v.y = -v.y;
        } else if (r == i) {
            v.x = rdiag[i];
        }
        X[e] = v;
        W[e] = make_double2(r == i ? 1.0 : 0.0, 0.0);
    }
    if (tid == 0) rotated = 0;
    __syncthreads();

    // one-sided Jacobi, round-robin pairs
    const int N = n + (n & 1), half = lane & 31, pair = tid >> 5;
    const double tol2 = kJacobiTol * kJacobiTol * n;
    int sweep = 0;
    for (; sweep < kJacobiSweeps && n > 1; ++sweep) {
        for (int round = 0; round < N - 1; ++round) {
            for (int pr = pair; pr < N / 2; pr += THREADS / 32) {
                int a = round + pr, b = round + N - 1 - pr;  // mod N - 1; pair 0 holds column N - 1
                a = pr == 0 ? N - 1 : a >= N - 1 ? a - (N - 1) : a;
                b = pr == 0 ? round : b >= N - 1 ? b - (N - 1) : b;
                if (a > b) {
                    const int q = a;
                    a = b;
                    b = q;
                }
                if (b >= n) continue;  // odd n: no partner this round
                double2 *xa = X + a * n, *xb = X + b * n, *wa = W + a * n, *wb = W + b * n;
                const bool in0 = half < n, in1 = half + 32 < n;
                const double2 z = make_double2(0, 0);
                double2 a0 = in0 ? xa[half] : z, b0 = in0 ? xb[half] : z;
                double2 a1 = in1 ? xa[half + 32] : z, b1 = in1 ? xb[half + 32] : z;
                double2 p0 = in0 ? wa[half] : z, q0 = in0 ? wb[half] : z;
                double2 p1 = in1 ? wa[half + 32] : z, q1 = in1 ? wb[half + 32] : z;
                const double na = half_all(a0.x * a0.x + a0.y * a0.y + a1.x * a1.x + a1.y * a1.y);
                const double nb = half_all(b0.x * b0.x + b0.y * b0.y + b1.x * b1.x + b1.y * b1.y);
                const double cr = half_all(a0.x * b0.x + a0.y * b0.y + a1.x * b1.x + a1.y * b1.y);
                const double ci = half_all(a0.x * b0.y - a0.y * b0.x + a1.x * b1.y - a1.y * b1.x);
                const double c2 = cr * cr + ci * ci;
                if (c2 > tol2 * na * nb && fmin(na, nb) > kJacobiZero) {
                    // d = |b|^2 - |a|^2, r = sqrt(d^2 + 4 |c|^2): cos^2 = (1 + |d| / r) / 2 and
                    // sin cos = |c| / r; the phase of c goes with the sine
                    const double d = nb - na, ir = rsqrt(d * d + 4.0 * c2);
                    const double cs2 = 0.5 + 0.5 * fabs(d) * ir, ic = rsqrt(cs2), cs = cs2 * ic;
                    const double f = copysign(ir * ic, d), sr = f * cr, si = -f * ci;
                    auto turn = [&](double2& u, double2& v) {  // (u, v) <- (cs u - s v, conj(s) u + cs v)
                        const double2 o = u;
                        u = make_double2(cs * o.x - (sr * v.x - si * v.y), cs * o.y - (sr * v.y + si * v.x));
                        v = make_double2(cs * v.x + (sr * o.x + si * o.y), cs * v.y + (sr * o.y - si * o.x));
                    };
                    turn(a0, b0);
                    turn(p0, q0);
                    if (in0) {
                        xa[half] = a0;
                        xb[half] = b0;
                        wa[half] = p0;
                        wb[half] = q0;
                    }
                    if (in1) {
                        turn(a1, b1);
                        turn(p1, q1);
                        xa[half + 32] = a1;
                        xb[half + 32] = b1;
                        wa[half + 32] = p1;
                        wb[half + 32] = q1;
                    }
                    if (half == 0) rotated = 1;
                }
            }
            __syncthreads();
        }
        const int again = rotated;
        __syncthreads();
        if (tid == 0) rotated = 0;
        if (!again) break;
        __syncthreads();
    }
    __syncthreads();
    const bool failed = sweep == kJacobiSweeps;

    // singular values in descending order
    for (int i = pair; i < n; i += THREADS / 32) {
        double s = 0;
        for (int r = half; r < n; r += 32) {
            const double2 v = X[i * n + r];
            s += v.x * v.x + v.y * v.y;
        }
        s = half_all(s);
        if (half == 0) nrm[i] = s > kJacobiZero ? sqrt(s) : 0.0;
    }
    __syncthreads();
    if (tid < n) {
        int rank = 0;
        for (int i = 0; i < n; ++i) rank += nrm[i] > nrm[tid] || (nrm[i] == nrm[tid] && i < tid);
        ord[rank] = tid;
        J.S[rank] = failed ? -1.0 : ldexp(nrm[tid], ex);
    }
    __syncthreads();
    // the short side's vectors x = Y / s
    for (int e = tid; e < n * n; e += THREADS) {
        const int k = e / n, r = e % n, o = ord[k];
        const double f = nrm[o] > 0 ? 1.0 / nrm[o] : amax > 0 ? 0.0 : 1.0;
        // (the value 0 is kept of a zero matrix only: any orthonormal vectors)
        const double2 v = amax > 0 ? X[o * n + r] : make_double2(r == k ? 1.0 : 0.0, 0.0);
        if (tall)
            J.Vh[e] = make_double2(f * v.x, -f * v.y);
        else
            J.U[r * n + k] = make_double2(f * v.x, f * v.y);
    }
    // the rotations in that order and the reflectors' scalars, for jacobi_apply_kernel
    for (int e = tid; e < n * n; e += THREADS) J.W[e] = W[ord[e / n] * n + e % n];
    if (tid < n) J.tau[tid] = tau[tid];
}

// The long side's vectors: column k of Q [W; 0] in one wave, the next reflector's entries loaded
// while this one's inner product is reduced.  The columns are spread over the CUs: in the
// decomposition's own workgroup they took as long as its reduction and rotations together.
template <int NT>
__global__ __launch_bounds__(64) void jacobi_apply_kernel(const SvdJob* __restrict__ jobs) {
    const SvdJob J = jobs[blockIdx.y];
    const bool tall = J.nr >= J.nc;
    const int n = tall ? J.nc : J.nr, m = tall ? J.nr : J.nc, k = blockIdx.x, lane = threadIdx.x;
    if (k >= n || (J.zero_ends && J.S[n - 1] == 0)) return;
    const double2* w = J.W + k * n;
    const double2* A = J.A;
    ColView<NT> c((tall ? J.T : J.Vh) + (int64_t)k * m, m, lane);
    auto out = [&](int i, double2& v) {
        if (tall)
            J.U[(int64_t)i * n + k] = v;
        else
            J.Vh[(int64_t)k * m + i] = make_double2(v.x, -v.y);
    };
    if constexpr (NT > 0) {
        double2 v[NT];
        auto load = [&](int j) {
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                const int i = lane + 64 * t;
                v[t] = make_double2(0, 0);
                if (i >= j && i < m) v[t] = A[(int64_t)j * m + i];
            }
        };
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const int i = lane + 64 * t;
            c.r[t] = i < n ? w[i] : make_double2(0, 0);
        }
        load(n - 1);
        for (int j = n - 1; j >= 0; --j) {
            const double2 tj = J.tau[j];
            double2 u[NT];
#pragma unroll
            for (int t = 0; t < NT; ++t) u[t] = v[t];
            if (j > 0) load(j - 1);
            double wr = 0, wi = 0;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                wr += u[t].x * c.r[t].x + u[t].y * c.r[t].y;
                wi += u[t].x * c.r[t].y - u[t].y * c.r[t].x;
            }
            wr = wave_all(wr);
            wi = wave_all(wi);
            const double gr = tj.x * wr - tj.y * wi, gi = tj.x * wi + tj.y * wr;
#pragma unroll
            for (int t = 0; t < NT; ++t) {
                c.r[t].x -= u[t].x * gr - u[t].y * gi;
                c.r[t].y -= u[t].x * gi + u[t].y * gr;
            }
        }
        c.each(0, false, out);
    } else {
        for (int i = lane; i < m; i += 64) c.p[i] = i < n ? w[i] : make_double2(0, 0);
        for (int j = n - 1; j >= 0; --j) {
            const double2 tj = J.tau[j];
            const double2* v = A + (int64_t)j * m;
            double wr = 0, wi = 0;
            c.each(j, false, [&](int i, double2& a) {
                const double2 u = v[i];
                wr += u.x * a.x + u.y * a.y;
                wi += u.x * a.y - u.y * a.x;
            });
            wr = wave_all(wr);
            wi = wave_all(wi);
            const double gr = tj.x * wr - tj.y * wi, gi = tj.x * wi + tj.y * wr;
            c.each(j, true, [&](int i, double2& a) {
                const double2 u = v[i];
                a.x -= u.x * gr - u.y * gi;
                a.y -= u.x * gi + u.y * gr;
            });
        }
        c.each(0, false, out);
    }
}

void launch_jacobi_svd(hipStream_t st, const SvdJob* jobs, int njobs, int nmax, int mmax) {
    if (njobs <= 0) return;
    const size_t lds = (size_t)2 * nmax * nmax * sizeof(double2);
    // a column's rows per lane; from nine up half the waves, for the registers
    const auto f = mmax <= 64     ? jacobi_svd_kernel<1, 1024>
                   : mmax <= 256  ? jacobi_svd_kernel<4, 1024>
                   : mmax <= 512  ? jacobi_svd_kernel<8, 1024>
                   : mmax <= 768  ? jacobi_svd_kernel<12, 512>
                   : mmax <= 1536 ? jacobi_svd_kernel<24, 512>
                                  : jacobi_svd_kernel<0, 1024>;
    const int threads = mmax > 512 && mmax <= 1536 ? 512 : 1024;
    KV_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(f), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)((size_t)2 * kJacobiMax * kJacobiMax * sizeof(double2))));
    hipLaunchKernelGGL(f, dim3(njobs), dim3(threads), lds, st, jobs);
    KV_HIP(hipGetLastError());
    const auto g = mmax <= 64     ? jacobi_apply_kernel<1>
                   : mmax <= 256  ? jacobi_apply_kernel<4>
                   : mmax <= 512  ? jacobi_apply_kernel<8>
                   : mmax <= 768  ? jacobi_apply_kernel<12>
                   : mmax <= 1536 ? jacobi_apply_kernel<24>
                                  : jacobi_apply_kernel<0>;
    hipLaunchKernelGGL(g, dim3(nmax, njobs), dim3(64), 0, st, jobs);
    KV_HIP(hipGetLastError());
}

// A[i ld + i] = (v, 0) for i in [from, to): the diagonal of a square matrix (either order).
__global__ __launch_bounds__(256) void set_diag_kernel(double2* __restrict__ A, int64_t ld, int from,
                                                       int to, double v) {
    for (int i = from + blockIdx.x * 256 + threadIdx.x; i < to; i += gridDim.x * 256)
        A[(int64_t)i * ld + i] = make_double2(v, 0.0);
}

void launch_set_diag(hipStream_t st, double2* A, int64_t ld, int from, int to, double v) {
    if (to <= from) return;
    hipLaunchKernelGGL(set_diag_kernel, dim3(ew_blocks(to - from)), dim3(256), 0, st, A, ld, from, to, v);
    KV_HIP(hipGetLastError());
}

// dst (n x n, row-major, ld n) = one triangle of src (ld lds), the other triangle zero:
// dst[i][j] = src[i * lds + j] where j <= i (lower) or j >= i (upper).
__global__ __launch_bounds__(256) void tri_copy_kernel(const double2* __restrict__ src, int64_t lds,
                                                       double2* __restrict__ dst, int n, int lower) {
    const int64_t total = (int64_t)n * n;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (int64_t)gridDim.x * 256) {
        const int i = (int)(e / n), j = (int)(e % n);
        const bool keep = lower ? j <= i : j >= i;
        dst[e] = keep ? src[(int64_t)i * lds + j] : make_double2(0.0, 0.0);
    }
}

void launch_tri_copy(hipStream_t st, const double2* src, int64_t lds, double2* dst, int n, bool lower) {
    if (n <= 0) return;
    hipLaunchKernelGGL(tri_copy_kernel, dim3(ew_blocks((int64_t)n * n)), dim3(256), 0, st, src, lds, dst, n,
                       lower ? 1 : 0);
    KV_HIP(hipGetLastError());
}

// ---- back-transformation of a Householder tridiagonalisation ------------------------
// Lower-triangle reduction Q^H A Q = T of a column-major n x n matrix: reflector i < n-1 is
// H_i = I - tau_i v_i v_i^H with v_i[r] = 0 for r <= i, 1 at r = i + 1 and A[i n + r] below.
// V (column-major, n rows, ncols >= n - 1 columns) receives every v_i explicitly; columns
// from n - 1 on are zero.
__global__ __launch_bounds__(256) void hh_explicit_kernel(const double2* __restrict__ A,
                                                          double2* __restrict__ V, int n,
                                                          int ncols) {
    const int64_t total = (int64_t)n * ncols;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (int64_t)gridDim.x * 256) {
        const int i = (int)(e / n), r = (int)(e % n);
        double2 v = make_double2(0.0, 0.0);
        if (i < n - 1) {
            if (r == i + 1)
                v.x = 1.0;
            else if (r > i + 1)
                v = A[e];
        }
        V[e] = v;
    }
}

void launch_hh_explicit(hipStream_t st, const double2* A, double2* V, int n, int ncols) {
    const int64_t total = (int64_t)n * ncols;
    if (total <= 0) return;
    hipLaunchKernelGGL(hh_explicit_kernel, dim3(ew_blocks(total)), dim3(256), 0, st, A, V, n, ncols);
    KV_HIP(hipGetLastError());
}

// ---- symmetric tridiagonal eigenproblem: divide and conquer --------------------------------
// All matrices of a bond together (sides up to kStedcMax): diagonal blocks of 8 by cyclic Jacobi
// in a wave each, then levels of merges, each one launch that deflates and solves the secular equations
// (one workgroup per merge) and one that multiplies the eigenvectors (32 x 32 tiles over all
// CUs).  Cuppen's splitting with the deflation of LAPACK's dlaed2, roots by Li's two-pole
// interpolation inside a bracket (LAPACK Working Note 89), vectors from the recomputed z of Gu and
// Eisenstat (SIAM J. Matrix Anal. Appl. 16 (1995)), which are orthonormal to rounding.
// Bound by latency: a root's iterations, and the deflation scan.  rocSOLVER's dstedc takes some
// twenty launches a level and one matrix at a time: 0.45 ms for a side of 128, 0.95 for 256; here a
// bond's matrices take 0.17 ms together at 128, of which the four merges' secular equations 0.11.
constexpr int kLeaf = 8;  // (blocks of 32 in 256 threads: 0.34 ms, longer than all merges)
constexpr double kEps = 1.1102230246251565e-16;

// Total order on (value, index), NaN included, so that a rank by counting is a permutation.
__device__ inline bool before(double a, int i, double b, int k) {
    const int64_t u = __double_as_longlong(a), v = __double_as_longlong(b);
    const int64_t x = u ^ (int64_t)((uint64_t)(u >> 63) >> 1), y = v ^ (int64_t)((uint64_t)(v >> 63) >> 1);
    return x < y || (x == y && i < k);
}

__device__ inline double rcp64(double x) {  // 1 / x to an ulp, no special cases
    double r = __builtin_amdgcn_rcp(x);
    r = fma(fma(-x, r, 1.0), r, r);
    return fma(fma(-x, r, 1.0), r, r);
}

// Leaves: block b of matrix blockIdx.y, after the split subtracted |e| on both sides of every
// block boundary; values ascending into d1, vectors into the block of Q.
__global__ __launch_bounds__(64) void stedc_leaf_kernel(const StedcJob* __restrict__ jobs) {
    __shared__ double A[kLeaf][kLeaf + 1], V[kLeaf][kLeaf + 1], cs[kLeaf / 2], sn[kLeaf / 2];
    __shared__ double val[kLeaf];
    __shared__ int pp[kLeaf / 2], qq[kLeaf / 2], live;
    const StedcJob J = jobs[blockIdx.y];
    const int lo = blockIdx.x * kLeaf, n = J.n, tid = threadIdx.x;
    if (lo >= n) return;
    const int m = min(kLeaf, n - lo);
    double big = 0;
    for (int i = tid; i < n; i += 64) big = fmax(big, fmax(fabs(J.d[i]), i + 1 < n ? fabs(J.e[i]) : 0.0));
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) big = fmax(big, __shfl_xor(big, s));
    big = fmax(big, 1e-300);
    const double sc = 1.0 / big;
    if (blockIdx.x == 0 && tid == 0) J.scale[0] = sc;
    for (int64_t e = (int64_t)lo * n + tid; e < (int64_t)(lo + m) * n; e += 64) J.Q1[e] = J.Q2[e] = 0.0;
    for (int e = tid; e < kLeaf * kLeaf; e += 64) {
        const int i = e / kLeaf, j = e % kLeaf;
        double v = 0;
        if (i < m && j < m) {
            if (i == j) {
                v = J.d[lo + i] * sc;
                if (i == 0 && lo > 0) v -= fabs(J.e[lo - 1] * sc);
                if (i == m - 1 && lo + m < n) v -= fabs(J.e[lo + m - 1] * sc);
            } else if (i == j + 1 || j == i + 1) {
                v = J.e[lo + min(i, j)] * sc;
            }
        }
        A[i][j] = v;
        V[i][j] = i == j ? 1.0 : 0.0;
    }
    __syncthreads();
    for (int sweep = 0; sweep < 20; ++sweep) {
        if (tid == 0) live = 0;
        __syncthreads();
        for (int round = 0; round < kLeaf - 1; ++round) {
            if (tid < kLeaf / 2) {
                int a = round + tid, b = round + kLeaf - 1 - tid;
                a = tid == 0 ? kLeaf - 1 : a >= kLeaf - 1 ? a - (kLeaf - 1) : a;
                b = tid == 0 ? round : b >= kLeaf - 1 ? b - (kLeaf - 1) : b;
                const int p = min(a, b), q = max(a, b);
                const double apq = A[p][q], app = A[p][p], aqq = A[q][q];
                double c = 1, s = 0;
                if (fabs(apq) > 0.5 * kEps * (fabs(app) + fabs(aqq)) && fabs(apq) > 1e-300) {
                    const double th = (aqq - app) / (2.0 * apq);
                    const double t = copysign(1.0 / (fabs(th) + sqrt(1.0 + th * th)), th);
                    c = 1.0 / sqrt(1.0 + t * t);
                    s = t * c;
                    // a rotation below the absolute accuracy of the block does not hold up the end
                    if (fabs(apq) > 1e-18) live = 1;
                }
                pp[tid] = p;
                qq[tid] = q;
                cs[tid] = c;
                sn[tid] = s;
            }
            __syncthreads();
            {  // columns p, q of A by one half of the wave, of V by the other
                const int k = (tid & 31) / kLeaf, r = tid % kLeaf, p = pp[k], q = qq[k];
                const double c = cs[k], s = sn[k];
                double(*M)[kLeaf + 1] = tid < 32 ? A : V;
                const double x = M[r][p], y = M[r][q];
                M[r][p] = c * x - s * y;
                M[r][q] = s * x + c * y;
            }
            __syncthreads();
            if (tid < 32) {  // rows
                const int k = tid / kLeaf, r = tid % kLeaf, p = pp[k], q = qq[k];
                const double c = cs[k], s = sn[k];
                const double x = A[p][r], y = A[q][r];
                A[p][r] = c * x - s * y;
                A[q][r] = s * x + c * y;
            }
            __syncthreads();
        }
        const int again = live;
        __syncthreads();
        if (!again) break;
    }
    if (tid < m) val[tid] = A[tid][tid];
    __syncthreads();
    if (tid < m) {
        int rank = 0;
        for (int i = 0; i < m; ++i) rank += before(val[i], i, val[tid], tid);
        J.d1[lo + rank] = val[tid];
        for (int i = 0; i < m; ++i) J.Q1[(int64_t)(lo + rank) * n + lo + i] = V[i][tid];
    }
}

// One merge of blocks [lo, mid) and [mid, hi) of width h: what becomes of every column.
__global__ __launch_bounds__(512) void stedc_merge_kernel(const StedcJob* __restrict__ jobs, int h, int flip) {
    __shared__ double d[kStedcMax], z[kStedcMax], dk[kStedcMax], zk[kStedcMax], tau[kStedcMax], zh[kStedcMax];
    __shared__ double rc[kStedcMax], rs[kStedcMax], red[16];
    __shared__ int ord[kStedcMax], col[kStedcMax], org[kStedcMax], rp[kStedcMax], rq[kStedcMax];
    __shared__ int K_s, nrot_s;
    const StedcJob J = jobs[blockIdx.y];
    const int n = J.n, lo = blockIdx.x * 2 * h, mid = min(lo + h, n), hi = min(lo + 2 * h, n), tid = threadIdx.x;
    if (lo >= n) return;
    const int N = hi - lo;
    const double* din = flip ? J.d2 : J.d1;
    double* dout = flip ? J.d1 : J.d2;
    double* Q = flip ? J.Q2 : J.Q1;
    if (mid >= hi) {  // no partner: every column stays
        if (tid == 0) J.kcount[lo / (2 * h)] = 0;
        for (int i = tid; i < N; i += 512) {
            dout[lo + i] = din[lo + i];
            J.src[lo + i] = lo + i;
            J.pos[lo + i] = lo + i;
        }
        return;
    }
    const double e = J.e[mid - 1] * J.scale[0], rho = 2.0 * fabs(e), inv2 = 0.70710678118654752440;
    double dm = 0, zm = 0;
    for (int i = tid; i < N; i += 512) {
        d[i] = din[lo + i];
        const double q = i < mid - lo ? Q[(int64_t)(lo + i) * n + mid - 1] : copysign(1.0, e) * Q[(int64_t)(lo + i) * n + mid];
        z[i] = q * inv2;
        dm = fmax(dm, fabs(d[i]));
        zm = fmax(zm, fabs(z[i]));
    }
#pragma unroll
    for (int s = 32; s > 0; s >>= 1) {
        dm = fmax(dm, __shfl_xor(dm, s));
        zm = fmax(zm, __shfl_xor(zm, s));
    }
    if ((tid & 63) == 0) {
        red[tid >> 6] = dm;
        red[8 + (tid >> 6)] = zm;
    }
    __syncthreads();
    for (int w = 0; w < 8; ++w) {
        dm = fmax(dm, red[w]);
        zm = fmax(zm, red[8 + w]);
    }
    const double tol = 8.0 * kEps * fmax(dm, zm);
    for (int i = tid; i < N; i += 512) {
        int rank = 0;
        for (int k = 0; k < N; ++k) rank += before(d[k], k, d[i], i);
        ord[rank] = i;
    }
    __syncthreads();
    for (int k = tid; k < N; k += 512) {
        tau[k] = d[ord[k]];
        zh[k] = z[ord[k]];
    }
    __syncthreads();
    // deflation along the ascending values (one thread: each decision depends on the one before)
    if (tid == 0) {
        int K = 0, nd = N, nrot = 0, pj = -1, no = ord[0];
        double dp = 0, zp = 0, dn = tau[0], zn = zh[0];
        for (int k = 0; k < N; ++k) {
            const int nj = no, k1 = min(k + 1, N - 1);
            double dj = dn, zj = zn;
            no = ord[k1];
            dn = tau[k1];
            zn = zh[k1];
            if (rho * fabs(zj) <= tol) {
                col[--nd] = nj;
                continue;
            }
            if (pj >= 0) {
                const double t2 = zp * zp + zj * zj;
                if (fabs((dj - dp) * zj * zp) <= tol * t2) {  // rotate zp away: its column is an eigenvector
                    const double ir = 1.0 / sqrt(t2), c = zj * ir, s = -zp * ir;
                    rp[nrot] = pj;
                    rq[nrot] = nj;
                    rc[nrot] = c;
                    rs[nrot++] = s;
                    d[pj] = dp * c * c + dj * s * s;
                    dj = dp * s * s + dj * c * c;
                    zj = t2 * ir;
                    col[--nd] = pj;
                } else {
                    dk[K] = dp;
                    zk[K] = zp;
                    col[K++] = pj;
                }
            }
            pj = nj;
            dp = dj;
            zp = zj;
        }
        if (pj >= 0) {
            dk[K] = dp;
            zk[K] = zp;
            col[K++] = pj;
        }
        K_s = K;
        nrot_s = nrot;
    }
    __syncthreads();
    const int K = K_s, nrot = nrot_s;
    // rotations, a row a thread; where one starts at the column that the last one ended at, its
    // value is carried over, and the loads of eight run together
    for (int r = lo + tid; nrot > 0 && r < hi; r += 512) {
        double carry = 0;
        for (int k0 = 0; k0 < nrot; k0 += 8) {
            double y[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) y[u] = Q[(int64_t)(lo + rq[min(k0 + u, nrot - 1)]) * n + r];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int k = k0 + u;
                if (k >= nrot) break;
                double* x = Q + (int64_t)(lo + rp[k]) * n + r;
                const double a = k > 0 && rp[k] == rq[k - 1] ? carry : *x;
                *x = rc[k] * a + rs[k] * y[u];
                carry = rc[k] * y[u] - rs[k] * a;
                if (k + 1 == nrot || rp[k + 1] != rq[k]) Q[(int64_t)(lo + rq[k]) * n + r] = carry;
            }
        }
    }
    // secular equation 1 / rho + sum_j z_j^2 / (d_j - x) = 0: root k between poles k and k + 1 (the
    // last one above the last pole), as an offset t from the nearer pole in a bracket (a, b) there;
    // first the root of the two nearest terms with the others as they are in the middle, then
    // steps of the same form fitted to the value and slopes of the two sides.  TPR lanes a root.
    constexpr int TPR = 2;
    const int sub = tid % TPR;
    const double irho = 1.0 / rho;
    for (int k = tid / TPR; k < K; k += 512 / TPR) {
        const bool last = k == K - 1;
        double zz = 0;
        if (last) {
            for (int j = sub; j < K; j += TPR) zz += zk[j] * zk[j];
            zz += __shfl_xor(zz, 1);
        }
        const double gap = last ? rho * zz : dk[k + 1] - dk[k];
        if (K == 1) {
            if (sub == 0) {
                tau[0] = gap;
                org[0] = 0;
            }
            continue;
        }
        const int sp = last ? k - 1 : k;  // the two poles of the interpolation: sp and sp + 1
        double psi, dpsi, phi, dphi;
        auto eval = [&](int s, double t) {  // the sums over poles <= sp and > sp at d_s + t
            psi = dpsi = phi = dphi = 0;
            const double o = dk[s];
            for (int j = sub; j < K; j += TPR) {
                const double r = rcp64((dk[j] - o) - t), w = zk[j] * zk[j] * r;
                if (j <= sp) {
                    psi += w;
                    dpsi += w * r;
                } else {
                    phi += w;
                    dphi += w * r;
                }
            }
            psi += __shfl_xor(psi, 1);
            dpsi += __shfl_xor(dpsi, 1);
            phi += __shfl_xor(phi, 1);
            dphi += __shfl_xor(dphi, 1);
        };
        int s = k;
        double t = 0.5 * gap, a = 0.0, b = gap;
        eval(s, t);
        double f = irho + psi + phi;
        const double z1 = zk[sp] * zk[sp], z2 = zk[sp + 1] * zk[sp + 1], del = dk[sp + 1] - dk[sp];
        const double c = f - z1 / ((dk[sp] - dk[s]) - t) - z2 / ((dk[sp + 1] - dk[s]) - t);
        if (!last && f < 0) {  // nearer to the upper pole
            s = k + 1;
            t = -0.5 * gap;
            a = t;
            b = 0.0;
        } else if (f < 0) {
            a = t;
        } else {
            b = t;
        }
        const double p1 = dk[sp] - dk[s], p2 = dk[sp + 1] - dk[s];
        double x;
        if (s == sp) {
            const double A = c * del + z1 + z2, B = z1 * del, D = sqrt(fabs(A * A - 4.0 * B * c));
            x = A > 0 ? 2.0 * B / (A + D) : (A - D) / (2.0 * c);
        } else {
            const double A = z1 + z2 - c * del, B = z2 * del, D = sqrt(fabs(A * A + 4.0 * B * c));
            x = last ? (A < 0 ? 2.0 * B / (D - A) : (A + D) / (2.0 * c))
                     : (A > 0 ? -2.0 * B / (A + D) : (A - D) / (2.0 * c));
        }
        if (x > a && x < b && x != t) t = x;
        eval(s, t);
        f = irho + psi + phi;
        for (int it = 0; it < 60; ++it) {
            const double df = dpsi + dphi;
            if (fabs(f) <= kEps * (8.0 * (fabs(psi) + fabs(phi) + irho) + fabs(t) * df)) break;
            if (f < 0)
                a = t;
            else
                b = t;
            const double d1 = p1 - t, d2 = p2 - t;
            double cc = f - d1 * dpsi - d2 * dphi;
            const double aa = (d1 + d2) * f - d1 * d2 * df, bb = d1 * d2 * f;
            const double disc = sqrt(fabs(aa * aa - 4.0 * bb * cc));
            double eta;
            if (last) {
                cc = fabs(cc);
                eta = aa >= 0 ? (aa + disc) / (2.0 * cc) : 2.0 * bb / (aa - disc);
            } else {
                eta = cc == 0 ? bb / aa : aa <= 0 ? (aa - disc) / (2.0 * cc) : 2.0 * bb / (aa + disc);
            }
            if (!(f * eta < 0)) eta = -f / df;
            double tn = t + eta;
            if (!(tn > a && tn < b)) tn = (f > 0 && a == 0) || (f < 0 && b == 0) ? t / 32 : 0.5 * (a + b);
            if (tn == t || !(tn > a && tn < b)) break;  // the bracket has closed
            t = tn;
            eval(s, t);
            f = irho + psi + phi;
        }
        if (sub == 0) {
            tau[k] = t;
            org[k] = s;
        }
    }
    __syncthreads();
    // z recomputed from the roots, so that they are exact eigenvalues of the modified matrix
    for (int j = tid / TPR; j < K; j += 512 / TPR) {
        double p = 1.0;
        for (int k = sub; k < K; k += TPR) {
            const double lam = (dk[org[k]] - dk[j]) + tau[k];  // lambda_k - d_j
            const double den = k < j ? dk[k] - dk[j] : k + 1 < K ? dk[k + 1] - dk[j] : 1.0;
            p *= lam / den;
        }
        p *= __shfl_xor(p, 1);
        if (sub == 0) zh[j] = copysign(sqrt(fabs(p)), zk[j]);
    }
    __syncthreads();
    for (int k = tid / TPR; k < K; k += 512 / TPR) {
        const double o = dk[org[k]], t = tau[k];
        double q = 0;
        for (int j = sub; j < K; j += TPR) {
            const double u = zh[j] / ((dk[j] - o) - t);
            q += u * u;
        }
        q += __shfl_xor(q, 1);
        const double f = 1.0 / sqrt(q);
        for (int j = sub; j < K; j += TPR) J.U[(int64_t)(lo + j) * n + lo + k] = f * (zh[j] / ((dk[j] - o) - t));
    }
    __syncthreads();
    // ascending order over roots and deflated values
    for (int i = tid; i < N; i += 512) z[i] = i < K ? dk[org[i]] + tau[i] : d[col[i]];
    __syncthreads();
    for (int i = tid; i < N; i += 512) {
        int rank = 0;
        for (int k = 0; k < N; ++k) rank += before(z[k], k, z[i], i);
        dout[lo + rank] = z[i];
        J.src[lo + i] = lo + col[i];
        J.pos[lo + i] = lo + rank;
    }
    if (tid == 0) J.kcount[lo / (2 * h)] = K;
}

// Eigenvectors of the merged blocks: column pos[k] = sum_j Q(:, src[j]) U(j, k) over the K roots, the
// deflated columns copied.  Workgroup (x, y, z): 32 rows x 32 columns of a block pair.
__global__ __launch_bounds__(256) void stedc_vectors_kernel(const StedcJob* __restrict__ jobs, int h, int flip) {
    __shared__ double As[32][33], Bs[32][33];
    const StedcJob J = jobs[blockIdx.z];
    const int n = J.n, tiles = (2 * h + 31) / 32;
    const int lo = blockIdx.y * 2 * h, hi = min(lo + 2 * h, n), N = hi - lo;
    const int r0 = (blockIdx.x / tiles) * 32, c0 = (blockIdx.x % tiles) * 32, tid = threadIdx.x;
    if (lo >= n || r0 >= N || c0 >= N) return;
    const double* Q = flip ? J.Q2 : J.Q1;
    double* out = flip ? J.Q1 : J.Q2;
    const int K = J.kcount[blockIdx.y];
    const int tx = tid & 31, ty = tid >> 5;
    double acc[4] = {0, 0, 0, 0};
    if (c0 < K) {
        for (int j0 = 0; j0 < K; j0 += 32) {
            for (int q = 0; q < 4; ++q) {
                const int i = ty + 8 * q, j = j0 + i;
                As[i][tx] = j < K && r0 + tx < N ? Q[(int64_t)J.src[lo + j] * n + lo + r0 + tx] : 0.0;
                Bs[i][tx] = j < K && c0 + tx < K ? J.U[(int64_t)(lo + j) * n + lo + c0 + tx] : 0.0;
            }
            __syncthreads();
            for (int j = 0; j < 32; ++j)
#pragma unroll
                for (int q = 0; q < 4; ++q) acc[q] += As[j][tx] * Bs[j][ty + 8 * q];
            __syncthreads();
        }
    }
    for (int q = 0; q < 4; ++q) {
        const int c = c0 + ty + 8 * q, r = r0 + tx;
        if (c < N && r < N) {
            const double v = c < K ? acc[q] : Q[(int64_t)J.src[lo + c] * n + lo + r];
            out[(int64_t)J.pos[lo + c] * n + lo + r] = v;
        }
    }
}

// Values scaled back, vectors to their place.
__global__ __launch_bounds__(256) void stedc_end_kernel(const StedcJob* __restrict__ jobs, int flip) {
    const StedcJob J = jobs[blockIdx.y];
    const int64_t nn = (int64_t)J.n * J.n;
    const double* Q = flip ? J.Q2 : J.Q1;
    const double* d = flip ? J.d2 : J.d1;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < nn; e += (int64_t)gridDim.x * 256) J.Z[e] = Q[e];
    if (blockIdx.x == 0)
        for (int i = threadIdx.x; i < J.n; i += 256) J.w[i] = d[i] / J.scale[0];
}

static_assert(kLeaf == 8, "the leaf kernel's lanes");

void launch_stedc(hipStream_t st, const StedcJob* jobs, int njobs, int nmax) {
    KV_REQUIRE(nmax >= 1 && nmax <= kStedcMax, ERR_INTERNAL, "stedc: side above kStedcMax");
    if (njobs <= 0) return;
    hipLaunchKernelGGL(stedc_leaf_kernel, dim3((nmax + kLeaf - 1) / kLeaf, njobs), dim3(64), 0, st, jobs);
    KV_HIP(hipGetLastError());
    int flip = 0;
    for (int h = kLeaf; h < nmax; h *= 2, flip ^= 1) {
        const int nm = (nmax + 2 * h - 1) / (2 * h), tiles = (2 * h + 31) / 32;
        hipLaunchKernelGGL(stedc_merge_kernel, dim3(nm, njobs), dim3(512), 0, st, jobs, h, flip);
        KV_HIP(hipGetLastError());
        hipLaunchKernelGGL(stedc_vectors_kernel, dim3(tiles * tiles, nm, njobs), dim3(256), 0, st, jobs, h, flip);
        KV_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(stedc_end_kernel, dim3((nmax * nmax + 1023) / 1024, njobs), dim3(256), 0, st, jobs, flip);
    KV_HIP(hipGetLastError());
}

// Columns [c0, c0 + k) of C (real, column-major, ld n) carried through the reflectors of A
// (LAPACK zhetrd('L') storage): Z = H_0 H_1 ... H_{n-2} C(:, c0:c0+k), column-major complex.
// A wave keeps HHC columns in registers (rows lane + 64 u) and applies the reflectors from the
// last to the first, the next one's entries loaded while this one's inner products are reduced:
// a latency-bound chain of n reductions, no barriers and one launch.  The blocked form (explicit
// V, S = V^H V, T, then three products a block) takes a dozen launches and a 1.2 us step per
// column of T (bond SVD of two 128-wide sectors 3.22 -> 2.82 ms, 200-wide 4.69 -> 4.39).
constexpr int HHC = 2;
template <int NU>
__global__ __launch_bounds__(64) void hh_apply_kernel(const double2* __restrict__ A, const double2* __restrict__ tau,
                                                      const double* __restrict__ C, int n, int c0, int k,
                                                      double2* __restrict__ Z) {
    const int lane = threadIdx.x, j0 = blockIdx.x * HHC;
    double2 z[HHC][NU], v[NU];
#pragma unroll
    for (int c = 0; c < HHC; ++c)
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const int r = lane + 64 * u;
            z[c][u] = make_double2(r < n && j0 + c < k ? C[(int64_t)(c0 + j0 + c) * n + r] : 0.0, 0.0);
        }
    auto load = [&](int i) {  // v_i: 1 at row i + 1, the stored tail below
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const int r = lane + 64 * u;
            v[u] = make_double2(r == i + 1 ? 1.0 : 0.0, 0.0);
            if (r > i + 1 && r < n) v[u] = A[(int64_t)i * n + r];
        }
    };
    double2 t = make_double2(0, 0);
    if (n > 1) {
        load(n - 2);
        t = tau[n - 2];
    }
    for (int i = n - 2; i >= 0; --i) {
        double2 w[NU];
        const double2 ti = t;
#pragma unroll
        for (int u = 0; u < NU; ++u) w[u] = v[u];
        if (i > 0) {
            load(i - 1);
            t = tau[i - 1];
        }
        double dr[HHC], di[HHC];
#pragma unroll
        for (int c = 0; c < HHC; ++c) {
            dr[c] = di[c] = 0;
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                dr[c] += w[u].x * z[c][u].x + w[u].y * z[c][u].y;
                di[c] += w[u].x * z[c][u].y - w[u].y * z[c][u].x;
            }
        }
#pragma unroll
        for (int c = 0; c < HHC; ++c) {
            dr[c] = lane_first(tree64(dr[c]));
            di[c] = lane_first(tree64(di[c]));
        }
#pragma unroll
        for (int c = 0; c < HHC; ++c) {
            const double gr = ti.x * dr[c] - ti.y * di[c], gi = ti.x * di[c] + ti.y * dr[c];
#pragma unroll
            for (int u = 0; u < NU; ++u) {
                z[c][u].x -= w[u].x * gr - w[u].y * gi;
                z[c][u].y -= w[u].x * gi + w[u].y * gr;
            }
        }
    }
#pragma unroll
    for (int c = 0; c < HHC; ++c)
#pragma unroll
        for (int u = 0; u < NU; ++u) {
            const int r = lane + 64 * u;
            if (r < n && j0 + c < k) Z[(int64_t)(j0 + c) * n + r] = z[c][u];
        }
}

void launch_hh_apply(hipStream_t st, const double2* A, const double2* tau, const double* C, int n, int c0, int k,
                     double2* Z) {
    KV_REQUIRE(n >= 1 && n <= kHhApplyMax, ERR_INTERNAL, "hh_apply: side above kHhApplyMax");
    if (k <= 0) return;
    const auto f = n <= 64 ? hh_apply_kernel<1> : n <= 128 ? hh_apply_kernel<2> : n <= 256 ? hh_apply_kernel<4>
                                                                                           : hh_apply_kernel<8>;
    hipLaunchKernelGGL(f, dim3((k + HHC - 1) / HHC), dim3(64), 0, st, A, tau, C, n, c0, k, Z);
    KV_HIP(hipGetLastError());
}

// Triangular factors of blocks of bw consecutive reflectors (forward, columnwise):
// H_{i0} ... H_{i0+w-1} = I - V_b T_b V_b^H with T_b(c,c) = tau_c and
// T_b(0:c, c) = -tau_c T_b(0:c, 0:c) S_b(0:c, c), S_b = V_b^H V_b.  S and T hold one bw x bw
// column-major matrix per block; entries of columns c >= w (past the last reflector) are 0.
// One workgroup per block; the upper triangle of T_b lives packed in LDS (column j at
// j (j + 1) / 2).  Each new column is a triangular matrix-vector product: row r is summed
// by kTfSplit threads over interleaved j, partial sums combined through LDS.  The next
// column of S is loaded into registers while the current column is formed, so the global
// load is off the column-to-column chain; two barriers per column.
constexpr int kTfactorMax = 128, kTfSplit = 4;
__global__ __launch_bounds__(kTfactorMax * kTfSplit) void hh_tfactor_kernel(
    const double2* __restrict__ S, const double2* __restrict__ tau, double2* __restrict__ T, int bw,
    int nref) {
    __shared__ double2 tp[kTfactorMax * (kTfactorMax + 1) / 2];
    __shared__ double2 sc[kTfactorMax], tl[kTfactorMax];
    __shared__ double2 part[kTfSplit][kTfactorMax];
    const int b = blockIdx.x;
    const int i0 = b * bw;
    const int w = min(bw, nref - i0);
    const int r = threadIdx.x % kTfactorMax, q = threadIdx.x / kTfactorMax;
    const double2* Sb = S + (int64_t)b * bw * bw;
    double2* Tb = T + (int64_t)b * bw * bw;
    const double2 zero2 = make_double2(0.0, 0.0);
    // prologue: taus, column 0 (tau_0), S(:, 1) into sc and S(:, 2) into registers
    double2 pre = zero2;
    if (q == 0) {
        double2 t = zero2;
        if (r < w) t = tau[i0 + r];
        tl[r] = t;
        if (r == 0 && w > 0) tp[0] = t;
        double2 s1 = zero2;
        if (r < 1 && 1 < w) s1 = Sb[(int64_t)1 * bw + r];
        sc[r] = s1;
        if (r < 2 && 2 < w) pre = Sb[(int64_t)2 * bw + r];
    }
    __syncthreads();
    for (int c = 1; c < w; ++c) {
        // partial of sum_{j=r}^{c-1} T(r, j) S(j, c) over j = r + q, r + q + kTfSplit, ...
        double sr = 0.0, si = 0.0;
        if (r < c) {
#pragma unroll 4
            for (int j = r + q; j < c; j += kTfSplit) {
                const double2 a = tp[j * (j + 1) / 2 + r], x = sc[j];
                sr += a.x * x.x - a.y * x.y;
                si += a.x * x.y + a.y * x.x;
            }
        }
        part[q][r] = make_double2(sr, si);
        __syncthreads();
        if (q == 0) {
            const double2 t = tl[c];
            if (r < c) {
                double ar = 0.0, ai = 0.0;
#pragma unroll
                for (int u = 0; u < kTfSplit; ++u) {
                    ar += part[u][r].x;
                    ai += part[u][r].y;
                }
                tp[c * (c + 1) / 2 + r] = make_double2(-(t.x * ar - t.y * ai), -(t.x * ai + t.y * ar));
            } else if (r == c) {
                tp[c * (c + 1) / 2 + c] = t;
            }
            // column c + 1 of S for the next step, and the load of column c + 2
            sc[r] = pre;
            pre = zero2;
            if (r < c + 2 && c + 2 < w) pre = Sb[(int64_t)(c + 2) * bw + r];
        }
        __syncthreads();  // column c and sc complete before they are read
    }
    for (int e = threadIdx.x; e < bw * bw; e += blockDim.x) {
        const int c = e / bw, rr = e % bw;
        double2 t = zero2;
        if (c < w && rr <= c) t = tp[c * (c + 1) / 2 + rr];
        Tb[e] = t;
    }
}

void launch_hh_tfactor(hipStream_t st, const double2* S, const double2* tau, double2* T, int nblocks,
                       int bw, int nref) {
    if (nblocks <= 0) return;
    KV_REQUIRE(bw >= 1 && bw <= kTfactorMax, ERR_ARG, "reflector block width must be in [1, 128]");
    KV_REQUIRE((int64_t)nblocks * bw >= nref && (int64_t)(nblocks - 1) * bw < nref, ERR_ARG,
               "reflector blocks do not cover the reflectors");
    hipLaunchKernelGGL(hh_tfactor_kernel, dim3(nblocks), dim3(kTfactorMax * kTfSplit), 0, st, S, tau, T, bw,
                       nref);
    KV_HIP(hipGetLastError());
}

// out[e] = sum_{p < np} part[p * n + e]  (split-K partial products summed).
// Bound by the partials' read (np x n elements from L2 / HBM); eight loads in flight per lane.
template <class T2>
__global__ __launch_bounds__(256) void sum_parts_kernel(const T2* __restrict__ part, int np,
                                                        int64_t n, T2* __restrict__ out,
                                                        const int* __restrict__ stop) {
    if (stop && *stop) return;
    using T = typename ScalarOf<T2>::T;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
        T re = 0, im = 0;
#pragma unroll 8
        for (int p = 0; p < np; ++p) {
            const T2 v = part[(int64_t)p * n + e];
            re += v.x;
            im += v.y;
        }
        T2 o;
        o.x = re;
        o.y = im;
        out[e] = o;
    }
}

template <class T2>
void launch_sum_parts(hipStream_t st, const T2* part, int np, int64_t n, T2* out, const int* stop) {
    if (n <= 0) return;
    hipLaunchKernelGGL(sum_parts_kernel<T2>, dim3(ew_blocks(n)), dim3(256), 0, st, part, np, n, out, stop);
    KV_HIP(hipGetLastError());
}
template void launch_sum_parts<double2>(hipStream_t, const double2*, int, int64_t, double2*, const int*);
template void launch_sum_parts<float2>(hipStream_t, const float2*, int, int64_t, float2*, const int*);

// Z[j n + i] = C[(c0 + j) ldc + i] for i < n, j < k (real columns to complex).
__global__ __launch_bounds__(256) void real_cols_kernel(const double* __restrict__ C, int ldc, int c0,
                                                        int k, int n, double2* __restrict__ Z) {
    const int64_t total = (int64_t)n * k;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (int64_t)gridDim.x * 256) {
        const int j = (int)(e / n), i = (int)(e % n);
        Z[e] = make_double2(C[(int64_t)(c0 + j) * ldc + i], 0.0);
    }
}

void launch_real_cols(hipStream_t st, const double* C, int ldc, int c0, int k, int n, double2* Z) {
    const int64_t total = (int64_t)n * k;
    if (total <= 0) return;
    hipLaunchKernelGGL(real_cols_kernel, dim3(ew_blocks(total)), dim3(256), 0, st, C, ldc, c0, k, n, Z);
    KV_HIP(hipGetLastError());
}


// ---- Householder tridiagonalisation (lower triangle, LAPACK storage) ----------------
// Batched reduction Q^H A Q = T of column-major n x n Hermitian matrices (one per grid.y),
// blocked by panels of kTrdPanel columns: within a panel column j is brought up to date by
// the panel's earlier reflectors (V) and their companions (W), reflected (larfg), and its
// companion W(:, i) = tau (A v - V (W^H v) - W (V^H v)) + alpha v formed from a matvec over
// the trailing matrix as it stood at the panel start; after the panel the trailing matrix
// takes the rank-2 update A -= V W^H + W V^H on both triangles.  A is kept fully Hermitian
// (both triangles) so the matvec is a set of independent column dot products.  On exit
// D = diag(T), E = subdiag(T), tau and the reflector tails below the subdiagonal of A follow
// LAPACK zhetrd('L').  VW holds V in columns [0, nb) and W in [nb, 2 nb) (column-major,
// n rows); q holds W^H v in [0, nb) and V^H v in [nb, 2 nb).

// Mirror the lower triangle of each column-major n x n matrix into its upper triangle
// (conjugated) and drop the imaginary part of the diagonal.  32 x 32 tiles, grid (T, T, batch).
__global__ __launch_bounds__(256) void herm_fill_kernel(double2* __restrict__ A, int n, int64_t stride) {
    const int ti = blockIdx.x, tj = blockIdx.y;  // source tile rows ti, columns tj (lower: ti >= tj)
    if (ti < tj) return;
    A += (int64_t)blockIdx.z * stride;
    __shared__ double2 t[32][33];
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int c = ty; c < 32; c += 8) {
        const int gr = ti * 32 + tx, gc = tj * 32 + c;
        if (gr < n && gc < n) t[c][tx] = A[(int64_t)gc * n + gr];
    }
    __syncthreads();
    for (int r = ty; r < 32; r += 8) {
        const int dc = ti * 32 + r, dr = tj * 32 + tx;  // destination (dr, dc) = conj(source (dc, dr))
        if (dc < n && dr < n) {
            const double2 v = t[tx][r];
            if (dc > dr)
                A[(int64_t)dc * n + dr] = make_double2(v.x, -v.y);
            else if (dc == dr)
                A[(int64_t)dc * n + dr] = make_double2(v.x, 0.0);
        }
    }
}

constexpr int kTrdRows = 64;  // rows per block of trd_column_kernel (x 4 slices of the panel index)
constexpr int kTrdReg = 8;    // rows per thread whose loads are issued together (256 threads: 2048 rows)

__device__ inline double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__device__ inline double2 cmulc(double2 a, double2 b) {  // a * conj(b)
    return make_double2(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y);
}
__device__ inline double2 wave_sum2(double2 v) {  // fixed butterfly over the 64 lanes
    for (int off = 32; off > 0; off >>= 1) {
        v.x += __shfl_xor(v.x, off, 64);
        v.y += __shfl_xor(v.y, off, 64);
    }
    return v;
}

// One column step of the panel, rows [j, n), grid (ceil((n - j) / 64), batch).
// prev: finish the companion of column j - 1 (local index i - 1): w' = tau_{j-1} (y - V q1 - W q2)
//   over the panel's columns before i - 1, alpha = -tau_{j-1} (w'^H v) / 2, W(:, i-1) = w' + alpha v.
// col: bring column j up to date with the panel's columns before i and reflect it (j < n - 1);
//   with v(j) = 1 the contribution of column i - 1 is -v conj(w'(j)) - w' - 2 Re(alpha) v.
// Each block writes its share of w'^H v; the last block to finish (ticket on count[b], which
// it resets) sums the shares in block order and does the O(n) tail: W, the final column, its
// norm, larfg and the reflector, with each thread's rows loaded together.
__global__ __launch_bounds__(256) void trd_column_kernel(double2* __restrict__ A, double2* __restrict__ VW,
                                                         const double2* __restrict__ y,
                                                         const double2* __restrict__ q, double* __restrict__ Dg,
                                                         double* __restrict__ Eg, double2* __restrict__ tau,
                                                         double2* __restrict__ part, unsigned* __restrict__ count,
                                                         int n, int j, int i, int nb, int prev, int col) {
    const int b = blockIdx.y;
    A += (int64_t)b * n * n;
    VW += (int64_t)b * n * 2 * nb;
    y += (int64_t)b * n;
    q += (int64_t)b * 2 * nb;
    Dg += (int64_t)b * n;
    Eg += (int64_t)b * n;
    tau += (int64_t)b * n;
    part += (int64_t)b * gridDim.x;
    const double2* V = VW;
    double2* W = VW + (int64_t)nb * n;
    const double2 zero2 = make_double2(0.0, 0.0);
    const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
    const int K = prev ? i - 1 : 0;  // panel columns with final companions
    __shared__ double2 vj[kTrdPanel], wj[kTrdPanel], q1[kTrdPanel], q2[kTrdPanel];
    __shared__ double2 rw[4][kTrdRows], rc[4][kTrdRows], red[kTrdRows];
    __shared__ double2 wpj_s, alpha_s, alf_s, scale_s;
    __shared__ double ssq[4];
    __shared__ int last;
    const double2 taup = prev ? tau[j - 1] : zero2;
    if (threadIdx.x < K) {
        vj[threadIdx.x] = V[(int64_t)threadIdx.x * n + j];
        wj[threadIdx.x] = W[(int64_t)threadIdx.x * n + j];
        q1[threadIdx.x] = q[threadIdx.x];
        q2[threadIdx.x] = q[nb + threadIdx.x];
    }
    const int r = j + blockIdx.x * kTrdRows + tx;
    double2 yr = zero2, ar = zero2, vr = zero2;
    if (ty == 0 && r < n) {
        if (prev) {
            yr = y[r];
            vr = V[(int64_t)(i - 1) * n + r];
        }
        if (col) ar = A[(int64_t)j * n + r];
    }
    __syncthreads();
    if (prev && threadIdx.x < 64) {  // w'(j), needed by every row of column j: one panel column per lane
        double2 t = zero2;
        if (threadIdx.x < K) {
            const double2 a = cmul(vj[threadIdx.x], q1[threadIdx.x]), c = cmul(wj[threadIdx.x], q2[threadIdx.x]);
            t = make_double2(a.x + c.x, a.y + c.y);
        }
        t = wave_sum2(t);
        if (threadIdx.x == 0) {
            const double2 yj = y[j];
            wpj_s = cmul(taup, make_double2(yj.x - t.x, yj.y - t.y));
        }
    }
    double2 sw = zero2, sc = zero2;
    if (r < n) {
        for (int k = ty; k < K; k += 4) {
            const double2 vk = V[(int64_t)k * n + r], wk = W[(int64_t)k * n + r];
            const double2 a = cmul(vk, q1[k]), c = cmul(wk, q2[k]);
            sw.x += a.x + c.x;
            sw.y += a.y + c.y;
            const double2 e = cmulc(vk, wj[k]), f = cmulc(wk, vj[k]);
            sc.x += e.x + f.x;
            sc.y += e.y + f.y;
        }
    }
    rw[ty][tx] = sw;
    rc[ty][tx] = sc;
    __syncthreads();
    if (ty == 0) {
        double2 d = zero2;
        if (r < n) {
            for (int t = 1; t < 4; ++t) {
                sw.x += rw[t][tx].x;
                sw.y += rw[t][tx].y;
                sc.x += rc[t][tx].x;
                sc.y += rc[t][tx].y;
            }
            double2 wp = zero2;
            if (prev) {
                wp = cmul(taup, make_double2(yr.x - sw.x, yr.y - sw.y));
                W[(int64_t)(i - 1) * n + r] = wp;
                d = cmulc(vr, wp);  // conj(wp) v
            }
            if (col) {
                double2 c0 = make_double2(ar.x - sc.x, ar.y - sc.y);
                if (prev) {
                    const double2 t2 = cmulc(vr, wpj_s);
                    c0.x -= t2.x + wp.x;
                    c0.y -= t2.y + wp.y;
                }
                A[(int64_t)j * n + r] = c0;
            }
        }
        d = wave_sum2(d);
        if (tx == 0) {
            part[blockIdx.x] = d;
            __threadfence();
            last = atomicAdd(&count[b], 1u) == gridDim.x - 1;
        }
    }
    __syncthreads();
    if (!last) return;
    __threadfence();
    // ---- tail, one block: rows [j, n) ----
    if (threadIdx.x < 64) {
        double2 d = zero2;
        if (prev)
            for (unsigned t = threadIdx.x; t < gridDim.x; t += 64) {
                d.x += part[t].x;
                d.y += part[t].y;
            }
        d = wave_sum2(d);
        if (threadIdx.x == 0) {
            alpha_s = prev ? cmul(make_double2(-0.5 * taup.x, -0.5 * taup.y), d) : zero2;
            alf_s = zero2;
            count[b] = 0u;
        }
    }
    __syncthreads();
    const double2 alpha = alpha_s;
    const double g2 = 2.0 * alpha.x;
    const int m = n - j;
    const bool spill = m > 256 * kTrdReg;  // rows beyond the registers go back through A
    double2 cv[kTrdReg];
    double s2 = 0.0;
    for (int base = 0; base < m; base += 256 * kTrdReg) {
        double2 vv[kTrdReg], ww[kTrdReg], cc[kTrdReg];
#pragma unroll
        for (int u = 0; u < kTrdReg; ++u) {
            const int rr = j + base + u * 256 + threadIdx.x;
            vv[u] = zero2;
            ww[u] = zero2;
            cc[u] = zero2;
            if (rr < n) {
                if (prev) {
                    vv[u] = V[(int64_t)(i - 1) * n + rr];
                    ww[u] = W[(int64_t)(i - 1) * n + rr];
                }
                if (col) cc[u] = A[(int64_t)j * n + rr];
            }
        }
#pragma unroll
        for (int u = 0; u < kTrdReg; ++u) {
            const int rr = j + base + u * 256 + threadIdx.x;
            if (rr >= n) continue;
            if (prev) {
                const double2 av = cmul(alpha, vv[u]);
                W[(int64_t)(i - 1) * n + rr] = make_double2(ww[u].x + av.x, ww[u].y + av.y);
            }
            if (col) {
                const double2 c = make_double2(cc[u].x - g2 * vv[u].x, cc[u].y - g2 * vv[u].y);
                if (base == 0) cv[u] = c;
                if (spill) A[(int64_t)j * n + rr] = c;
                if (rr == j) Dg[j] = c.x;
                if (rr == j + 1) alf_s = c;
                if (rr >= j + 2) s2 += c.x * c.x + c.y * c.y;
            }
        }
    }
    if (!col || j >= n - 1) return;
    {
        double2 t = wave_sum2(make_double2(s2, 0.0));
        if (tx == 0) ssq[ty] = t.x;
    }
    __syncthreads();
    if (threadIdx.x == 0) {  // larfg: H^H [alpha; x] = [beta; 0], H = I - tau v v^H, v = [1; x / (alpha - beta)]
        const double2 a = alf_s;
        const double xn2 = ((ssq[0] + ssq[1]) + ssq[2]) + ssq[3];
        double beta, tr = 0.0, ti = 0.0;
        double2 z = make_double2(1.0, 0.0);
        if (xn2 == 0.0 && a.y == 0.0) {
            beta = a.x;
        } else {
            beta = -copysign(sqrt(a.x * a.x + a.y * a.y + xn2), a.x);
            tr = (beta - a.x) / beta;
            ti = -a.y / beta;
            const double zr = a.x - beta, zi = a.y, z2 = zr * zr + zi * zi;
            z = make_double2(zr / z2, -zi / z2);
        }
        Eg[j] = beta;
        tau[j] = make_double2(tr, ti);
        scale_s = z;
        A[(int64_t)j * n + j + 1] = make_double2(beta, 0.0);
        VW[(int64_t)i * n + j + 1] = make_double2(1.0, 0.0);
    }
    __syncthreads();
    const double2 scl = scale_s;
    for (int base = 0; base < m; base += 256 * kTrdReg) {
#pragma unroll
        for (int u = 0; u < kTrdReg; ++u) {
            const int rr = j + base + u * 256 + threadIdx.x;
            if (rr < j + 2 || rr >= n) continue;
            const double2 v = cmul(base == 0 ? cv[u] : A[(int64_t)j * n + rr], scl);
            A[(int64_t)j * n + rr] = v;
            VW[(int64_t)i * n + rr] = v;
        }
    }
}

// y[c] = sum_{r >= s} conj(A(r, c)) v(r) for c in [s, n) (= (A v)(c), A Hermitian), then
// q[k] = W(:, k)^H v and q[nb + k] = V(:, k)^H v over rows [s, n) for k < i, with v = V(:, i).
// Two outputs per block of 256 threads, the rows spread over the block with each thread's
// loads issued together; grid (ceil((n - s + 2 i) / 2), batch).
__global__ __launch_bounds__(256) void trd_matvec_kernel(const double2* __restrict__ A,
                                                         const double2* __restrict__ VW, double2* __restrict__ y,
                                                         double2* __restrict__ q, int n, int s, int i, int nb) {
    const int b = blockIdx.y;
    A += (int64_t)b * n * n;
    VW += (int64_t)b * n * 2 * nb;
    y += (int64_t)b * n;
    q += (int64_t)b * 2 * nb;
    const int m = n - s, ntask = m + 2 * i;
    const int t0 = blockIdx.x * 2;
    const bool two = t0 + 1 < ntask;
    auto colp = [&](int t) -> const double2* {
        if (t < m) return A + (int64_t)(s + t) * n;
        t -= m;
        return t < i ? VW + (int64_t)(nb + t) * n : VW + (int64_t)(t - i) * n;  // W(:, t) or V(:, t - i)
    };
    const double2* c0 = colp(t0);
    const double2* c1 = two ? colp(t0 + 1) : c0;
    const double2* v = VW + (int64_t)i * n;
    double2 a0 = make_double2(0.0, 0.0), a1 = make_double2(0.0, 0.0);
    for (int base = s; base < n; base += 256 * kTrdReg) {
        double2 vv[kTrdReg], x0[kTrdReg], x1[kTrdReg];
#pragma unroll
        for (int u = 0; u < kTrdReg; ++u) {
            const int r = base + u * 256 + threadIdx.x;
            vv[u] = make_double2(0.0, 0.0);
            x0[u] = vv[u];
            x1[u] = vv[u];
            if (r < n) {
                vv[u] = v[r];
                x0[u] = c0[r];
                x1[u] = c1[r];
            }
        }
#pragma unroll
        for (int u = 0; u < kTrdReg; ++u) {
            const double2 e = cmulc(vv[u], x0[u]), f = cmulc(vv[u], x1[u]);  // conj(x) v
            a0.x += e.x;
            a0.y += e.y;
            a1.x += f.x;
            a1.y += f.y;
        }
    }
    a0 = wave_sum2(a0);
    a1 = wave_sum2(a1);
    __shared__ double2 red[2][4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) {
        red[0][wave] = a0;
        red[1][wave] = a1;
    }
    __syncthreads();
    if (threadIdx.x < 2 && (threadIdx.x == 0 || two)) {
        const int t = t0 + threadIdx.x;
        double2 acc = red[threadIdx.x][0];
        for (int w = 1; w < 4; ++w) {
            acc.x += red[threadIdx.x][w].x;
            acc.y += red[threadIdx.x][w].y;
        }
        if (t < m)
            y[s + t] = acc;
        else if (t - m < i)
            q[t - m] = acc;
        else
            q[nb + t - m - i] = acc;
    }
}

// The columns before the last kTrdRegMax of a Householder tridiagonalisation in zhetrd('L')'s
// form, Hermitian matrices up to kTrdSmallMax wide, one 768-thread workgroup per matrix (column-major, both triangles
// valid, as herm_fill leaves them).  Unblocked, with each step's rank-2 update fused into the
// next step's matrix-vector product: after column j's reflector v_j and y_j = A v_j,
//   w_j = tau_j y_j - (tau_j / 2) (tau_j y_j)^H v_j v_j,
//   column j + 1 brought up to date (A -= v_j w_j^H + w_j v_j^H on it) and reflected by
//   larfg's formulas (v_{j+1}, tau_{j+1}, beta = E[j+1]; the reflector's tail stored below
//   the subdiagonal of column j + 1 and beta on it),
//   one pass over A(j+2:, j+2:) applying the same update and forming y_{j+1} = A v_{j+1}
//   (as a combination of columns, exact for the Hermitian A the updates keep).
// Ends at column `end` (0 < end < n).
// D, E, tau and the stored reflectors are hetrd_lower's (the back-transformation reads them).
constexpr int kTrdSmallThreads = 768;
__global__ __launch_bounds__(kTrdSmallThreads) void trd_small_kernel(double2* __restrict__ A, int n, int end,
                                                                     double* __restrict__ Dg, double* __restrict__ Eg,
                                                                     double2* __restrict__ tau) {
    constexpr int NW = kTrdSmallThreads / 64, RU = kTrdSmallMax / 64;
    const int b = blockIdx.x;
    A += (int64_t)b * n * n;
    Dg += (int64_t)b * n;
    Eg += (int64_t)b * n;
    tau += (int64_t)b * n;
    __shared__ double2 vbuf[2][kTrdSmallMax], w0[kTrdSmallMax], y[kTrdSmallMax], col[kTrdSmallMax];
    __shared__ double2 part[NW][kTrdSmallMax];
    __shared__ double2 red2[NW];
    __shared__ double red1[NW];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const double2 zero2 = make_double2(0.0, 0.0);
    if (n <= 0) return;
    // larfg on col[j + 1 ..) (every thread the same arithmetic from the reduced norm): beta into
    // E and the subdiagonal, tau, the reflector into v (rows >= j + 1, v(j + 1) = 1) and below
    // the subdiagonal of column j.  Returns tau_j; ends synchronised.
    auto reflect = [&](int j, double2* v, double s2) -> double2 {
        for (int off = 32; off > 0; off >>= 1) s2 += __shfl_xor(s2, off, 64);
        if (lane == 0) red1[wv] = s2;
        __syncthreads();
        double xn2 = 0.0;
        for (int q = 0; q < NW; ++q) xn2 += red1[q];
        const double2 a = col[j + 1];
        double beta, tr = 0.0, ti = 0.0;
        double2 z = make_double2(1.0, 0.0);
        if (xn2 == 0.0 && a.y == 0.0) {
            beta = a.x;
        } else {
            beta = -copysign(sqrt(a.x * a.x + a.y * a.y + xn2), a.x);
            tr = (beta - a.x) / beta;
            ti = -a.y / beta;
            const double zr = a.x - beta, zi = a.y, z2 = zr * zr + zi * zi;
            z = make_double2(zr / z2, -zi / z2);
        }
        if (tid == 0) {
            Eg[j] = beta;
            tau[j] = make_double2(tr, ti);
            A[(int64_t)j * n + j + 1] = make_double2(beta, 0.0);
        }
        for (int r = tid; r < n; r += kTrdSmallThreads) {
            double2 vr = zero2;
            if (r == j + 1) {
                vr = make_double2(1.0, 0.0);
            } else if (r > j + 1) {
                vr = cmul(col[r], z);
                A[(int64_t)j * n + r] = vr;
            }
            v[r] = vr;
        }
        __syncthreads();
        return make_double2(tr, ti);
    };
    // y = A(s:, s:) v over rows and columns >= s, with the pending update (vp, w0) applied to
    // A(s:, s:) first and written back when `upd`; each lane's rows of a column are loaded
    // together before they are used
    // y = A(s:, s:) v over rows and columns >= s as a combination of columns (A is Hermitian,
    // so no reduction across lanes is needed): lane rows s + lane + 64 u, wave columns
    // s + wv CG + g + NW CG t; the pending update (vp, w0) is applied to A(s:, s:) first and
    // written back when `upd`.  The waves' partial vectors are summed in wave order.
    auto pass = [&](int s, const double2* v, const double2* vp, bool upd) {
        // columns per wave whose loads are issued before the first store (2 at 12 waves: 168 VGPRs,
        // no spills; 4 at 8 waves)
        constexpr int CG = kTrdSmallThreads > 512 ? 2 : 4;
        double2 acc[RU];
#pragma unroll
        for (int u = 0; u < RU; ++u) acc[u] = zero2;
        for (int c0 = s + wv * CG; c0 < n; c0 += NW * CG) {
            double2 a[CG][RU];
#pragma unroll
            for (int g = 0; g < CG; ++g)
#pragma unroll
                for (int u = 0; u < RU; ++u) {
                    const int r = s + lane + 64 * u, c = c0 + g;
                    a[g][u] = zero2;
                    if (r < n && c < n) a[g][u] = A[(int64_t)c * n + r];
                }
#pragma unroll
            for (int g = 0; g < CG; ++g) {
                const int c = c0 + g;
                if (c >= n) break;  // uniform over the wave
                const double2 wc = upd ? w0[c] : zero2, vc = upd ? vp[c] : zero2, xc = v[c];
#pragma unroll
                for (int u = 0; u < RU; ++u) {
                    const int r = s + lane + 64 * u;
                    if (r < n) {
                        double2 x = a[g][u];
                        if (upd) {
                            const double2 p = cmulc(vp[r], wc), q = cmulc(w0[r], vc);  // v(r) conj(w(c)) + w(r) conj(v(c))
                            x = make_double2(x.x - p.x - q.x, x.y - p.y - q.y);
                            A[(int64_t)c * n + r] = x;
                        }
                        const double2 e = cmul(x, xc);
                        acc[u].x += e.x;
                        acc[u].y += e.y;
                    }
                }
            }
        }
#pragma unroll
        for (int u = 0; u < RU; ++u) {
            const int r = s + lane + 64 * u;
            if (r < n) part[wv][r] = acc[u];
        }
        __syncthreads();
        for (int r = s + tid; r < n; r += kTrdSmallThreads) {
            double2 t = part[0][r];
            for (int q = 1; q < NW; ++q) {
                t.x += part[q][r].x;
                t.y += part[q][r].y;
            }
            y[r] = t;
        }
        __syncthreads();
    };
    // column 0
    double s2 = 0.0;
    for (int r = tid; r < n; r += kTrdSmallThreads) {
        const double2 x = A[r];
        col[r] = x;
        if (r >= 2) s2 += x.x * x.x + x.y * x.y;
    }
    if (tid == 0) Dg[0] = A[0].x;
    if (n == 1) return;
    __syncthreads();
    double2 tj = reflect(0, vbuf[0], s2);
    pass(1, vbuf[0], vbuf[0], false);
    for (int j = 0; j + 1 < n; ++j) {
        const double2* v0 = vbuf[j & 1];
        double2* v1 = vbuf[(j + 1) & 1];
        // alpha = -(tau/2) (tau y)^H v over rows >= j + 1
        double2 d = zero2;
        for (int r = j + 1 + tid; r < n; r += kTrdSmallThreads) {
            const double2 e = cmulc(v0[r], cmul(tj, y[r]));  // conj(tau y) v
            d.x += e.x;
            d.y += e.y;
        }
        d = wave_sum2(d);
        if (lane == 0) red2[wv] = d;
        __syncthreads();
        double2 t = zero2;
        for (int q = 0; q < NW; ++q) {
            t.x += red2[q].x;
            t.y += red2[q].y;
        }
        const double2 al = cmul(make_double2(-0.5 * tj.x, -0.5 * tj.y), t);
        for (int r = j + 1 + tid; r < n; r += kTrdSmallThreads) {
            const double2 x = cmul(tj, y[r]), av = cmul(al, v0[r]);
            w0[r] = make_double2(x.x + av.x, x.y + av.y);
        }
        __syncthreads();
        // column j + 1, up to date, and the norm of its tail
        const int c1 = j + 1;
        if (c1 == end) {  // the rest is trd_reg_kernel's: brought up to date
            for (int c = c1 + wv; c < n; c += NW)
                for (int r = c1 + lane; r < n; r += 64) {
                    const double2 a = A[(int64_t)c * n + r], p = cmulc(v0[r], w0[c]), q = cmulc(w0[r], v0[c]);
                    A[(int64_t)c * n + r] = make_double2(a.x - p.x - q.x, a.y - p.y - q.y);
                }
            break;
        }
        const double2 wc = w0[c1], vc = v0[c1];
        s2 = 0.0;
        for (int r = c1 + tid; r < n; r += kTrdSmallThreads) {
            const double2 a = A[(int64_t)c1 * n + r];
            const double2 p = cmulc(v0[r], wc), q = cmulc(w0[r], vc);
            const double2 x = make_double2(a.x - p.x - q.x, a.y - p.y - q.y);
            col[r] = x;
            if (r == c1) Dg[c1] = x.x;
            if (r >= c1 + 2) s2 += x.x * x.x + x.y * x.y;
        }
        if (c1 + 1 >= n) break;
        __syncthreads();
        tj = reflect(c1, v1, s2);
        pass(c1 + 1, v1, v0, true);
    }
}

// The same for a matrix of up to kTrdRegMax (its corner, when trd_small_kernel has done the columns
// before it), held in the registers of one 512-thread workgroup: waves 1 to 7 have columns
// w - 1 + 7 t, lane l rows l and l + 64.  The first wave alone does what is serial, its
// reductions by DPP: from the waves' parts of y it forms w, and while the others apply the update
// it brings the next column up to date and reflects it; then the others form y.  Column scalars
// come by readlane (LDS broadcasts would take as long as the arithmetic).
// Bound by that chain, 2.5 us a column: a side of 128 takes 0.32 ms (0.78 by trd_small_kernel, which
// reads and writes the matrix through L2 in every column; 0.43 with all eight waves in turn doing the
// chain, update and product behind two barriers), a side of 132 0.38 with its first columns (0.80).
constexpr int kTrdRegMax = 128;
__device__ inline double lane_get(double v, int l) {
    const uint64_t u = (uint64_t)__double_as_longlong(v);
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)u, l), hi = __builtin_amdgcn_readlane((uint32_t)(u >> 32), l);
    return __longlong_as_double((int64_t)(((uint64_t)hi << 32) | lo));
}
__device__ inline double2 lane_get2(double2 v, int l) { return make_double2(lane_get(v.x, l), lane_get(v.y, l)); }

__global__ __launch_bounds__(512) void trd_reg_kernel(double2* __restrict__ A, int ld, int j0, double* __restrict__ Dg,
                                                      double* __restrict__ Eg, double2* __restrict__ tau) {
    constexpr int NW = 7, CT = (kTrdRegMax + NW - 1) / NW;
    const int n = ld - j0;
    A += (int64_t)blockIdx.x * ld * ld + (int64_t)j0 * (ld + 1);
    Dg += (int64_t)blockIdx.x * ld + j0;
    Eg += (int64_t)blockIdx.x * ld + j0;
    tau += (int64_t)blockIdx.x * ld + j0;
    __shared__ double2 vs[2][kTrdRegMax], ws[kTrdRegMax], cs[kTrdRegMax], part[NW][kTrdRegMax];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6) - 1;
    const double2 zero2 = make_double2(0.0, 0.0);
    // z - v conj(w)
    auto sub_mulc = [](double2 z, double2 v, double2 w) {
        return make_double2(fma(-v.y, w.y, fma(-v.x, w.x, z.x)), fma(v.x, w.y, fma(-v.y, w.x, z.y)));
    };
    if (wv >= 0) {
        double2 a[CT][2];
#pragma unroll
        for (int t = 0; t < CT; ++t)
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                const int r = lane + 64 * u, c = wv + NW * t;
                a[t][u] = zero2;
                if (r < n && c < n && c > 0) a[t][u] = A[(int64_t)c * ld + r];
            }
        const int cl = min(wv + NW * (lane % CT), kTrdRegMax - 1);
        for (int j = 0; j + 1 < n; ++j) {
            __syncthreads();  // v of column j is there
            const double2* vj = vs[j & 1];
            const double2 xs = vj[cl];
            double2 acc[2] = {zero2, zero2};
#pragma unroll
            for (int t = 0; t < CT; ++t) {
                const int c = wv + NW * t;
                if (c <= j || c >= n) continue;
                const double2 xc = lane_get2(xs, t);
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    acc[u].x = fma(-a[t][u].y, xc.y, fma(a[t][u].x, xc.x, acc[u].x));
                    acc[u].y = fma(a[t][u].y, xc.x, fma(a[t][u].x, xc.y, acc[u].y));
                }
                if (c == j + 1) {
                    cs[lane] = a[t][0];
                    cs[lane + 64] = a[t][1];
                }
            }
            part[wv][lane] = acc[0];
            part[wv][lane + 64] = acc[1];
            __syncthreads();
            double2 vr[2], wr[2];
            for (int u = 0; u < 2; ++u) vr[u] = vj[lane + 64 * u];
            __syncthreads();  // w of column j is there
            const double2 pw = ws[cl];
            for (int u = 0; u < 2; ++u) wr[u] = ws[lane + 64 * u];
#pragma unroll
            for (int t = 0; t < CT; ++t) {
                const int c = wv + NW * t;
                if (c <= j + 1 || c >= n) continue;
                const double2 vc = lane_get2(xs, t), wc = lane_get2(pw, t);
#pragma unroll
                for (int u = 0; u < 2; ++u) a[t][u] = sub_mulc(sub_mulc(a[t][u], vr[u], wc), wr[u], vc);
            }
        }
        return;
    }
    // larfg on the column x (rows lane, lane + 64) below row j, as trd_small_kernel's reflect
    double2 v[2] = {zero2, zero2}, x[2], tj = zero2;
    auto reflect = [&](int j) {
        double s2 = 0.0;
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (lane + 64 * u >= j + 2) s2 += x[u].x * x[u].x + x[u].y * x[u].y;
        const double xn2 = wave_all(s2);
        const int l1 = (j + 1) & 63;
        const double2 al = lane_get2(j + 1 < 64 ? x[0] : x[1], l1);
        double beta, tr = 0.0, ti = 0.0;
        double2 z = make_double2(1.0, 0.0);
        if (xn2 == 0.0 && al.y == 0.0) {
            beta = al.x;
        } else {
            beta = -copysign(sqrt(al.x * al.x + al.y * al.y + xn2), al.x);
            tr = (beta - al.x) / beta;
            ti = -al.y / beta;
            const double zr = al.x - beta, zi = al.y, z2 = zr * zr + zi * zi;
            z = make_double2(zr / z2, -zi / z2);
        }
        tj = make_double2(tr, ti);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int r = lane + 64 * u;
            v[u] = r == j + 1 ? make_double2(1.0, 0.0) : r > j + 1 ? cmul(x[u], z) : zero2;
            vs[j & 1][r] = v[u];
            if (r > j && r < n) A[(int64_t)j * ld + r] = r == j + 1 ? make_double2(beta, 0.0) : v[u];
        }
        if (lane == 0) {
            Eg[j] = beta;
            tau[j] = tj;
        }
    };
#pragma unroll
    for (int u = 0; u < 2; ++u) x[u] = lane + 64 * u < n ? A[lane + 64 * u] : zero2;
    if (lane == 0) Dg[0] = x[0].x;
    if (n > 1) reflect(0);
    for (int j = 0; j + 1 < n; ++j) {
        __syncthreads();
        __syncthreads();  // y's parts and column j + 1 are there
        double2 y[2], d = zero2;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int r = lane + 64 * u;
            double2 t = part[0][r];
#pragma unroll
            for (int q = 1; q < NW; ++q) {
                t.x += part[q][r].x;
                t.y += part[q][r].y;
            }
            y[u] = r > j ? cmul(tj, t) : zero2;
            x[u] = cs[r];
            const double2 e = cmulc(v[u], y[u]);  // conj(tau y) v
            d.x += e.x;
            d.y += e.y;
        }
        d = make_double2(wave_all(d.x), wave_all(d.y));
        const double2 al = cmul(make_double2(-0.5 * tj.x, -0.5 * tj.y), d);
        double2 w[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const double2 av = cmul(al, v[u]);
            w[u] = make_double2(y[u].x + av.x, y[u].y + av.y);
            ws[lane + 64 * u] = w[u];
        }
        __syncthreads();
        const int c1 = j + 1, l1 = c1 & 63;
        const double2 wc = lane_get2(c1 < 64 ? w[0] : w[1], l1), vc = lane_get2(c1 < 64 ? v[0] : v[1], l1);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            x[u] = sub_mulc(sub_mulc(x[u], v[u], wc), w[u], vc);
            if (lane + 64 * u == c1) Dg[c1] = x[u].x;
        }
        if (c1 + 1 < n) reflect(c1);
    }
}

void launch_trd_small(hipStream_t st, double2* A, int n, double* D, double* E, double2* tau, int batch) {
    KV_REQUIRE(n >= 1 && n <= kTrdSmallMax && batch >= 1, ERR_INTERNAL, "trd_small: side above kTrdSmallMax");
    const int j0 = std::max(n - kTrdRegMax, 0);
    if (j0 > 0) {
        hipLaunchKernelGGL(trd_small_kernel, dim3(batch), dim3(kTrdSmallThreads), 0, st, A, n, j0, D, E, tau);
        KV_HIP(hipGetLastError());
    }
    hipLaunchKernelGGL(trd_reg_kernel, dim3(batch), dim3(512), 0, st, A, n, j0, D, E, tau);
    KV_HIP(hipGetLastError());
}

void launch_herm_fill(hipStream_t st, double2* A, int n, int batch) {
    if (n <= 0 || batch <= 0) return;
    const int T = (n + 31) / 32;
    hipLaunchKernelGGL(herm_fill_kernel, dim3(T, T, batch), dim3(256), 0, st, A, n, (int64_t)n * n);
    KV_HIP(hipGetLastError());
}

int trd_column_blocks(int n, int j) { return (n - j + kTrdRows - 1) / kTrdRows; }

void launch_trd_column(hipStream_t st, double2* A, double2* VW, const double2* y, const double2* q, double* D,
                       double* E, double2* tau, double2* part, unsigned* count, int n, int j, int i, int nb,
                       bool prev, bool col, int batch) {
    KV_REQUIRE(nb <= kTrdPanel && i <= nb && j >= 0 && j < n && (prev ? i >= 1 : i == 0) && j - i >= 0, ERR_INTERNAL,
               "trd_column: bad step");
    hipLaunchKernelGGL(trd_column_kernel, dim3(trd_column_blocks(n, j), batch), dim3(256), 0, st, A, VW, y, q, D,
                       E, tau, part, count, n, j, i, nb, prev ? 1 : 0, col ? 1 : 0);
    KV_HIP(hipGetLastError());
}

void launch_trd_matvec(hipStream_t st, const double2* A, const double2* VW, double2* y, double2* q, int n, int s,
                       int i, int nb, int batch) {
    KV_REQUIRE(s >= 1 && s < n && i >= 0 && i < nb && nb <= kTrdPanel, ERR_INTERNAL, "trd_matvec: bad step");
    const int ntask = n - s + 2 * i;
    hipLaunchKernelGGL(trd_matvec_kernel, dim3((ntask + 1) / 2, batch), dim3(256), 0, st, A, VW, y, q, n, s, i,
                       nb);
    KV_HIP(hipGetLastError());
}

// ---- block subspace route of the bond SVD --------------------------------------------
// Randomised range finding on a sector matrix (Halko, Martinsson and Tropp, SIAM Review 53
// (2011), algorithms 4.3/4.4 with Rayleigh-Ritz): a seeded random start block, Cholesky QR
// orthonormalisation with rank-deficient columns dropped, and the Ritz residual check.

// splitmix64 output function (Steele, Lea and Flood, OOPSLA 2014): a bijective 64-bit mix.
__device__ inline uint64_t mix64(uint64_t z) {
    z += 0x9e3779b97f4a7c15ull;
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ull;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebull;
    return z ^ (z >> 31);
}

// p[e] = (u, v) uniform in [-1, 1)^2, a function of (seed, e) only.
__global__ __launch_bounds__(256) void rand_fill_kernel(double2* __restrict__ p, int64_t n, uint64_t seed) {
    const uint64_t s = mix64(seed);
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < n; e += (int64_t)gridDim.x * 256) {
        const uint64_t a = mix64(s ^ (uint64_t)(2 * e)), b = mix64(s ^ (uint64_t)(2 * e + 1));
        p[e] = make_double2((double)(a >> 11) * 0x1.0p-52 - 1.0, (double)(b >> 11) * 0x1.0p-52 - 1.0);
    }
}

void launch_rand_fill(hipStream_t st, double2* p, int64_t n, uint64_t seed) {
    if (n <= 0) return;
    const int blocks = (int)std::min<int64_t>((n + 255) / 256, 4096);
    hipLaunchKernelGGL(rand_fill_kernel, dim3(blocks), dim3(256), 0, st, p, n, seed);
    KV_HIP(hipGetLastError());
}

__device__ inline double wave_max(double v) {
    for (int off = 32; off > 0; off >>= 1) v = fmax(v, __shfl_xor(v, off, 64));
    return v;
}

__device__ inline double2 cfma_conj(double2 acc, double2 a, double2 b) {  // acc + conj(a) b
    return make_double2(acc.x + a.x * b.x + a.y * b.y, acc.y + a.x * b.y - a.y * b.x);
}
__device__ inline double2 cfma(double2 acc, double2 a, double2 b) {  // acc + a b
    return make_double2(acc.x + a.x * b.x - a.y * b.y, acc.y + a.x * b.y + a.y * b.x);
}

// Largest real diagonal entry of each batched matrix (the Cholesky drop threshold's scale),
// read before any panel step overwrites S.  One workgroup per matrix.
__global__ __launch_bounds__(256) void diag_max_kernel(const double2* __restrict__ S, const int* __restrict__ sizes,
                                                       int ld, int64_t stride, double* __restrict__ dmax) {
    const int b = blockIdx.x, n = sizes[b];
    S += (int64_t)b * stride;
    __shared__ double red[4];
    double mx = 0.0;
    for (int i = threadIdx.x; i < n; i += 256) mx = fmax(mx, S[(int64_t)i * ld + i].x);
    mx = wave_max(mx);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    if (threadIdx.x == 0) dmax[b] = fmax(fmax(red[0], red[1]), fmax(red[2], red[3]));
}

// Left-looking blocked Cholesky S = R^H R with T = R^{-1}, panel k in two launches.
// Shared by both: 32 x 32 tile sums over rows of R (or T) staged through LDS in 32-row
// chunks, the four waves taking every fourth row and each lane a 4 x 4 block, the waves'
// partial tiles added in wave order.
struct CholTiles {
    double2 At[kCholLeftNB][kCholLeftNB + 1], Bt[kCholLeftNB][kCholLeftNB + 1];
    double2 red[3][kCholLeftNB][kCholLeftNB + 1];
};

// acc (this lane's 4 x 4 block of a 32 x 32 tile) += sum over rows i in [i_begin, i_end) of
// op(A)(i, r) B(i, c), with A(i, r) = S[i ld + a_col + r] (conj, arows = false) or
// T[(a_row + r) ld + i] (arows = true), B(i, c) = S[i ld + b_col + c] for c < bw; then the
// waves' blocks are added into wave 0's.
__device__ __forceinline__ void chol_tile_sum(CholTiles& L, double2 (&acc)[4][4], const double2* __restrict__ S,
                                     const double2* __restrict__ T, int ld, int i_begin, int i_end, int a_col,
                                     int a_row, bool arows, int aw, int b_col, int bw) {
    constexpr int NB = kCholLeftNB;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int r4 = (lane >> 3) * 4, c4 = (lane & 7) * 4;
    const double2 zero2 = make_double2(0.0, 0.0);
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y) acc[x][y] = zero2;
    // the next chunk's operands are loaded into registers while the current one is summed
    constexpr int NQ = NB * NB / 256;
    double2 pa[NQ], pb[NQ];
    auto fetch = [&](int i0) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int e = tid + 256 * q, ii = e / NB, cc = e % NB;
            pa[q] = zero2;
            pb[q] = zero2;
            if (arows)
                pa[q] = T[(int64_t)(a_row + ii) * ld + i0 + cc];  // A^T staged: At[r][i]
            else if (cc < aw)
                pa[q] = S[(int64_t)(i0 + ii) * ld + a_col + cc];
            if (cc < bw) pb[q] = S[(int64_t)(i0 + ii) * ld + b_col + cc];
        }
    };
    if (i_begin >= i_end) return;  // uniform over the workgroup
    fetch(i_begin);
    for (int i0 = i_begin; i0 < i_end; i0 += NB) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int e = tid + 256 * q;
            L.At[e / NB][e % NB] = pa[q];
            L.Bt[e / NB][e % NB] = pb[q];
        }
        __syncthreads();
        if (i0 + NB < i_end) fetch(i0 + NB);
        for (int ii = wv; ii < NB; ii += 4) {
            double2 av[4], bv[4];
#pragma unroll
            for (int x = 0; x < 4; ++x) {
                av[x] = arows ? L.At[r4 + x][ii] : L.At[ii][r4 + x];
                bv[x] = L.Bt[ii][c4 + x];
            }
#pragma unroll
            for (int x = 0; x < 4; ++x)
#pragma unroll
                for (int y = 0; y < 4; ++y)
                    acc[x][y] = arows ? cfma(acc[x][y], av[x], bv[y]) : cfma_conj(acc[x][y], av[x], bv[y]);
        }
        __syncthreads();
    }
    if (wv > 0)
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
            for (int y = 0; y < 4; ++y) L.red[wv - 1][r4 + x][c4 + y] = acc[x][y];
    __syncthreads();
    if (wv == 0)
#pragma unroll
        for (int q = 0; q < 3; ++q)
#pragma unroll
            for (int x = 0; x < 4; ++x)
#pragma unroll
                for (int y = 0; y < 4; ++y) {
                    const double2 v = L.red[q][r4 + x][c4 + y];
                    acc[x][y].x += v.x;
                    acc[x][y].y += v.y;
                }
    __syncthreads();
}

// Launch A of panel k, one workgroup per matrix: C_kk = S_kk - R_{<k,k}^H R_{<k,k}, its
// factor with the rank-tolerant pivot rule (a pivot at or below tau * dmax drops its column:
// R's row and T's row and column are zero; live flags), and its inverse Di, into T's tile
// (k, k) and Rd[b][k].  The factor is right-looking in LDS with all threads; the inverse of
// the triangular factor by recursive doubling: T_AC = -T_A R_AC T_C for pairs of diagonal
// blocks of 1, 2, 4, 8 and 16.
__global__ __launch_bounds__(256) void chol_diag_kernel(const double2* __restrict__ S, const int* __restrict__ sizes,
                                                        int ld, int64_t stride, double tau,
                                                        int* __restrict__ live, const double* __restrict__ dmax,
                                                        double2* __restrict__ T, double2* __restrict__ Rd, int k) {
    constexpr int NB = kCholLeftNB;
    const int b = blockIdx.x, n = sizes[b];
    const int p0 = k * NB;
    if (p0 >= n) return;  // uniform over the workgroup
    const int w = min(NB, n - p0);
    S += (int64_t)b * stride;
    T += (int64_t)b * stride;
    live += (int64_t)b * ld;
    Rd += ((int64_t)b * ((ld + NB - 1) / NB) + k) * NB * NB;
    const double thr = tau * dmax[b];
    __shared__ CholTiles L;
    __shared__ double2 Dg[NB][NB + 1], Ti[NB][NB + 1], Rf[NB][NB + 1];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int r4 = (lane >> 3) * 4, c4 = (lane & 7) * 4;
    const double2 zero2 = make_double2(0.0, 0.0);
    double2 ak[4][4];
    chol_tile_sum(L, ak, S, T, ld, 0, p0, p0, 0, false, w, p0, w);
    if (wv == 0)
#pragma unroll
        for (int x = 0; x < 4; ++x)
#pragma unroll
            for (int y = 0; y < 4; ++y) {
                const int r = r4 + x, c = c4 + y;
                double2 v = zero2;
                if (r < w && c < w && c >= r) {
                    const double2 sv = S[(int64_t)(p0 + r) * ld + p0 + c];
                    v = make_double2(sv.x - ak[x][y].x, sv.y - ak[x][y].y);
                }
                Dg[r][c] = v;
                Rf[r][c] = zero2;
            }
    __syncthreads();
    // factor, right-looking, all threads, one phase per pivot: a thread keeps column tid % 32 of
    // rows tid / 32 + 8 q in registers and updates them with row kk unscaled over the pivot; row
    // kk + 1, then final, goes to LDS for the next phase.  R's rows (Dg's over sqrt(piv)) are
    // formed after the last one, so that a phase waits for a reciprocal and not for a root and a
    // division (with both in each phase, all rows read back from LDS, and both kinds of tile in one
    // workgroup of the panel's second launch: 31 and 19 us for the two launches of a panel in
    // blocks 132 wide, 37 and 25 us 256 wide; now 24 and 15, 29 and 18).
    constexpr int NQ = NB * NB / 256;
    static_assert(NB == 32, "the factor's rows and columns per thread");
    const int c = tid % NB, i0 = tid / NB;
    double2 z[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) z[q] = Dg[i0 + 8 * q][c];
    __syncthreads();
    unsigned lv = 0u;
    for (int kk = 0; kk < w; ++kk) {
        const double piv = Dg[kk][kk].x;
        const double2 y = Dg[kk][c];
        const bool lk = piv > thr && piv > 0.0;  // NaN is not live
        const double rp = lk ? rcp64(piv) : 0.0;
        lv |= lk ? 1u << kk : 0u;
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            const int i = i0 + 8 * q;
            if (8 * q + 7 <= kk) continue;  // uniform
            if (i > kk && c >= i && c < w) {
                const double2 x = Dg[kk][i];
                if (lk) z[q] = make_double2(z[q].x - (x.x * y.x + x.y * y.y) * rp, z[q].y - (x.x * y.y - x.y * y.x) * rp);
                if (i == kk + 1) Dg[i][c] = z[q];
            }
        }
        __syncthreads();
    }
    for (int e = tid; e < NB * NB; e += 256) {
        const int i = e / NB, c = e % NB;
        if (i < w && c >= i && c < w) {  // R
            const double sp = (lv >> i) & 1u ? sqrt(Dg[i][i].x) : 0.0, ri = sp > 0.0 ? 1.0 / sp : 0.0;
            Rf[i][c] = c == i ? make_double2(sp, 0.0) : make_double2(Dg[i][c].x * ri, Dg[i][c].y * ri);
        }
    }
    __syncthreads();
    // Ti = diag(1 / R_ii) over live indices
    for (int e = tid; e < NB * NB; e += 256) {
        const int i = e / NB, c = e % NB;
        Ti[i][c] = (i == c && i < w && ((lv >> i) & 1u)) ? make_double2(1.0 / Rf[i][i].x, 0.0) : zero2;
    }
    __syncthreads();
    // recursive doubling: for pairs (A = [p, p+s), C = [p+s, p+2s)): M = R_AC T_C, T_AC = -T_A M
    // (M in Dg, free after the factor)
#pragma unroll
    for (int s = 1; s < NB; s *= 2) {
        const int per = s * s, tot = (NB / (2 * s)) * per;  // outputs per pair, all pairs
        for (int e = tid; e < tot; e += 256) {
            const int pr = e / per, rr = (e % per) / s, cc = e % s, p = pr * 2 * s;
            double2 m = zero2;
#pragma unroll
            for (int t = 0; t < s; ++t)
                if (t <= cc) m = cfma(m, Rf[p + rr][p + s + t], Ti[p + s + t][p + s + cc]);
            Dg[p + rr][p + s + cc] = m;
        }
        __syncthreads();
        for (int e = tid; e < tot; e += 256) {
            const int pr = e / per, rr = (e % per) / s, cc = e % s, p = pr * 2 * s;
            double2 m = zero2;
#pragma unroll
            for (int t = 0; t < s; ++t)
                if (t >= rr) m = cfma(m, Ti[p + rr][p + t], Dg[p + t][p + s + cc]);
            Ti[p + rr][p + s + cc] = make_double2(-m.x, -m.y);
        }
        __syncthreads();
    }
    for (int e = tid; e < NB * NB; e += 256) {
        const int i = e / NB, c = e % NB;
        Rd[e] = Ti[i][c];
        if (i < w && c < w) T[(int64_t)(p0 + i) * ld + p0 + c] = Ti[i][c];
    }
    if (tid < w) live[p0 + tid] = (lv >> tid) & 1u;
}

// Launch B of panel k, grid (ceil(nmax / 32), batch), one of np - 1 tiles a workgroup: for 0 < j <
// npk (panels from k on) R's tile (k, k + j) = Di^H (S_kc - R_{<k,k}^H R_{<k,c}) into S and a zero
// tile (k + j, k) into T; for j < k T's tile (j, k) = -(T_{j, j..k-1} R_{j..k-1, k}) Di.
// Tiles of S and T written here are read by no other workgroup of the launch.
__global__ __launch_bounds__(256) void chol_panel_kernel(double2* __restrict__ S, const int* __restrict__ sizes,
                                                         int ld, int64_t stride, double2* __restrict__ T,
                                                         const double2* __restrict__ Rd, int k) {
    constexpr int NB = kCholLeftNB;
    const int b = blockIdx.y, n = sizes[b];
    const int p0 = k * NB;
    if (p0 >= n) return;  // uniform over the workgroup
    const int w = min(NB, n - p0);
    const int npk = (n - p0 + NB - 1) / NB;
    const bool off = (int)blockIdx.x < npk - 1, inv = !off && (int)blockIdx.x < npk - 1 + k;
    const int j = off ? blockIdx.x + 1 : blockIdx.x - (npk - 1);
    if (!off && !inv) return;  // uniform over the workgroup
    S += (int64_t)b * stride;
    T += (int64_t)b * stride;
    Rd += ((int64_t)b * ((ld + NB - 1) / NB) + k) * NB * NB;
    __shared__ CholTiles L;
    __shared__ double2 Di[NB][NB + 1], Ct[NB][NB + 1];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int r4 = (lane >> 3) * 4, c4 = (lane & 7) * 4;
    const double2 zero2 = make_double2(0.0, 0.0);
    for (int e = tid; e < NB * NB; e += 256) Di[e / NB][e % NB] = Rd[e];
    const int r = tid >> 3, cq = (tid & 7) * 4;
    if (off) {
        const int c0 = p0 + j * NB, wc = min(NB, n - c0);
        double2 ac[4][4];
        chol_tile_sum(L, ac, S, T, ld, 0, p0, p0, 0, false, w, c0, wc);
        if (wv == 0)
#pragma unroll
            for (int x = 0; x < 4; ++x)
#pragma unroll
                for (int y = 0; y < 4; ++y) {
                    const int rr = r4 + x, c = c4 + y;
                    double2 v = zero2;
                    if (rr < w && c < wc) {
                        const double2 sv = S[(int64_t)(p0 + rr) * ld + c0 + c];
                        v = make_double2(sv.x - ac[x][y].x, sv.y - ac[x][y].y);
                    }
                    Ct[rr][c] = v;
                }
        __syncthreads();
        double2 yv[4] = {zero2, zero2, zero2, zero2};
#pragma unroll 4
        for (int m = 0; m <= r; ++m) {
            const double2 d = Di[m][r];
#pragma unroll
            for (int q = 0; q < 4; ++q) yv[q] = cfma_conj(yv[q], d, Ct[m][cq + q]);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int c = cq + q;
            if (r < w && c < wc) S[(int64_t)(p0 + r) * ld + c0 + c] = yv[q];
            if (c < w && r < wc) T[(int64_t)(c0 + r) * ld + p0 + c] = zero2;
        }
    }
    if (inv) {
        const int R0 = j * NB;
        double2 xa[4][4];
        chol_tile_sum(L, xa, S, T, ld, R0, p0, 0, R0, true, NB, p0, w);
        if (wv == 0)
#pragma unroll
            for (int x = 0; x < 4; ++x)
#pragma unroll
                for (int y = 0; y < 4; ++y) Ct[r4 + x][c4 + y] = xa[x][y];
        __syncthreads();
        double2 yv[4] = {zero2, zero2, zero2, zero2};
#pragma unroll 4
        for (int m = 0; m < cq + 4; ++m) {
            const double2 d = Ct[r][m];
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (m <= cq + q) yv[q] = cfma(yv[q], d, Di[m][cq + q]);
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
            if (cq + q < w) T[(int64_t)(R0 + r) * ld + p0 + cq + q] = make_double2(-yv[q].x, -yv[q].y);
    }
}

void launch_chol_left(hipStream_t st, double2* S, const int* sizes, int nmax, int ld, int64_t stride, double tau,
                      int* live, double* dmax, double2* T, double2* Rd, int batch) {
    KV_REQUIRE(nmax <= ld && batch >= 1, ERR_INTERNAL, "chol_left: side above the leading dimension");
    hipLaunchKernelGGL(diag_max_kernel, dim3(batch), dim3(256), 0, st, S, sizes, ld, stride, dmax);
    KV_HIP(hipGetLastError());
    const int np = (nmax + kCholLeftNB - 1) / kCholLeftNB;
    for (int k = 0; k < np; ++k) {
        hipLaunchKernelGGL(chol_diag_kernel, dim3(batch), dim3(256), 0, st, S, sizes, ld, stride, tau, live, dmax, T,
                           Rd, k);
        KV_HIP(hipGetLastError());
        hipLaunchKernelGGL(chol_panel_kernel, dim3(np, batch), dim3(256), 0, st, S, sizes, ld, stride, T, Rd, k);
        KV_HIP(hipGetLastError());
    }
}

// Column c of Y (n x ld, row-major) for every c < ld with live[c] == 0: seeded uniform
// complex values scaled so the column's squared norm is about dmax[0] (E|u|^2 = 2/3).
__global__ __launch_bounds__(256) void refill_cols_kernel(double2* __restrict__ Y, int n, int ld,
                                                          const int* __restrict__ live,
                                                          const double* __restrict__ dmax, uint64_t seed) {
    const uint64_t s = mix64(seed);
    const double f = sqrt(1.5 * fmax(dmax[0], 0.0) / (double)n);
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < (int64_t)n * ld; e += (int64_t)gridDim.x * 256) {
        const int c = (int)(e % ld);
        if (live[c]) continue;
        const uint64_t a = mix64(s ^ (uint64_t)(2 * e)), b = mix64(s ^ (uint64_t)(2 * e + 1));
        Y[e] = make_double2(f * ((double)(a >> 11) * 0x1.0p-52 - 1.0), f * ((double)(b >> 11) * 0x1.0p-52 - 1.0));
    }
}

void launch_refill_cols(hipStream_t st, double2* Y, int n, int ld, const int* live, const double* dmax,
                        uint64_t seed) {
    const int64_t total = (int64_t)n * ld;
    if (total <= 0) return;
    const int blocks = (int)std::min<int64_t>((total + 255) / 256, 4096);
    hipLaunchKernelGGL(refill_cols_kernel, dim3(blocks), dim3(256), 0, st, Y, n, ld, live, dmax, seed);
    KV_HIP(hipGetLastError());
}

// part[y kc + j] = sum over rows [y rows_per, (y + 1) rows_per) of |G[r][j] - theta_j Z[r][j]|^2
// (row-major G and Z, ld ldg and ldz).  grid (ceil(kc / 64), chunks), 4 row slices per block.
__global__ __launch_bounds__(256) void resid_cols_kernel(const double2* __restrict__ G, int ldg,
                                                         const double2* __restrict__ Z, int ldz,
                                                         const double* __restrict__ theta, int n, int kc,
                                                         int rows_per, double* __restrict__ part) {
    const int l = threadIdx.x & 63, sl = threadIdx.x >> 6;
    const int j = blockIdx.x * 64 + l;
    const int r0 = blockIdx.y * rows_per, r1 = min(n, r0 + rows_per);
    __shared__ double red[4][64];
    double s = 0.0;
    if (j < kc) {
        const double t = theta[j];
        for (int r = r0 + sl; r < r1; r += 4) {
            const double2 g = G[(int64_t)r * ldg + j], z = Z[(int64_t)r * ldz + j];
            const double dx = g.x - t * z.x, dy = g.y - t * z.y;
            s += dx * dx + dy * dy;
        }
    }
    red[sl][l] = s;
    __syncthreads();
    if (sl == 0 && j < kc) part[(int64_t)blockIdx.y * kc + j] = (red[0][l] + red[1][l]) + (red[2][l] + red[3][l]);
}

void launch_resid_cols(hipStream_t st, const double2* G, int ldg, const double2* Z, int ldz, const double* theta,
                       int n, int kc, int rows_per, double* part) {
    if (n <= 0 || kc <= 0) return;
    const int chunks = (n + rows_per - 1) / rows_per;
    hipLaunchKernelGGL(resid_cols_kernel, dim3((kc + 63) / 64, chunks), dim3(256), 0, st, G, ldg, Z, ldz, theta, n,
                       kc, rows_per, part);
    KV_HIP(hipGetLastError());
}

// ---- overlap over matching block pairs, and the allocation-free entry point's scratch -----

__global__ __launch_bounds__(256) void dotc_pairs_partial_kernel(const double2* __restrict__ x,
                                                                 const double2* __restrict__ y,
                                                                 const DotPair* __restrict__ pairs, int npairs,
                                                                 double* __restrict__ part) {
    __shared__ double sr[256], si[256];
    double re = 0, im = 0;
    for (int p = 0; p < npairs; ++p) {
        const DotPair d = pairs[p];
        for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < d.size; e += (int64_t)gridDim.x * 256) {
            const double2 a = x[d.x_off + e], b = y[d.y_off + e];
            re += a.x * b.x + a.y * b.y;  // conj(a) * b
            im += a.x * b.y - a.y * b.x;
        }
    }
    sr[threadIdx.x] = re;
    si[threadIdx.x] = im;
    __syncthreads();
    for (int s = 128; s > 0; s >>= 1) {
        if ((int)threadIdx.x < s) {
            sr[threadIdx.x] += sr[threadIdx.x + s];
            si[threadIdx.x] += si[threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = sr[0];
        part[2 * blockIdx.x + 1] = si[0];
    }
}

void launch_dotc_pairs(hipStream_t st, const double2* x, const double2* y, const DotPair* pairs, int npairs,
                       int64_t total, double* part, double2* out) {
    const int nb = red_blocks(total);  // every block writes its partial, also with no pairs
    hipLaunchKernelGGL(dotc_pairs_partial_kernel, dim3(nb), dim3(256), 0, st, x, y, pairs, npairs, part);
    KV_HIP(hipGetLastError());
    hipLaunchKernelGGL(reduce2_final_kernel, dim3(1), dim3(256), 0, st, part, nb, reinterpret_cast<double*>(out), 2);
    KV_HIP(hipGetLastError());
}

// The allocation-free entry point's scratch.  In host code `scratch` names a host-side
// stand-in, not device memory: only the address hipGetSymbolAddress returns for the
// current device may be handed to kernels and copies.
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::mutex& scratch_mutex() {
    static std::mutex m;
    return m;
}
void* scratch_ptr[kMaxDevices] = {nullptr};
}  // namespace

void noalloc_scratch_init(int device) {
    KV_REQUIRE(device >= 0 && device < kMaxDevices, ERR_ARG, "device index out of range");
    std::lock_guard<std::mutex> g(scratch_mutex());
    if (scratch_ptr[device]) return;
    int cur = -1;
    KV_HIP(hipGetDevice(&cur));
    KV_REQUIRE(cur == device, ERR_INTERNAL, "noalloc scratch: device is not current");
    void* p = nullptr;
    KV_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    KV_REQUIRE(p != nullptr, ERR_HIP, "hipGetSymbolAddress returned no address for the scratch");
    scratch_ptr[device] = p;
}

void* noalloc_scratch(int device) {
    KV_REQUIRE(device >= 0 && device < kMaxDevices, ERR_ARG, "device index out of range");
    std::lock_guard<std::mutex> g(scratch_mutex());
    KV_REQUIRE(scratch_ptr[device] != nullptr, ERR_INTERNAL, "noalloc scratch not initialised on this device");
    return scratch_ptr[device];
}

}  // namespace kv
