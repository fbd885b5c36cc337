// Contraction planners: turn the block structures of the operands into device work
// lists (grouped-GEMM tiles, MPO-fold tasks, permutation tasks).  Host-only C++ (no
// HIP), so the plans can be checked on a CPU against the oracle.
//
// A plan is built once per bond and reused for every Lanczos matvec on that bond; the
// executors in product.h upload its arrays to the device once.
#pragma once

#include <array>
#include <cmath>
#include <map>
#include <utility>
#include <vector>

#include "../kv_types.h"
#include "layout.h"

namespace kv {

inline int op_code(char op) {
    if (op == 'N') return 0;
    if (op == 'T') return 1;
    if (op == 'C') return 2;
    throw Error(ERR_ARG, std::string("bad op code ") + op);
}

// Output tiles of a group list for tile config cfg (kGemmConfigs), row-major per group.
inline std::vector<GemmTile> cut_tiles(const std::vector<GemmGroup>& groups, int cfg) {
    const int bm = kGemmConfigs[cfg].bm, bn = kGemmConfigs[cfg].bn;
    std::vector<GemmTile> t;
    for (int gi = 0; gi < (int)groups.size(); ++gi) {
        const int tm = (groups[gi].m + bm - 1) / bm, tn = (groups[gi].n + bn - 1) / bn;
        for (int a = 0; a < tm; ++a)
            for (int b = 0; b < tn; ++b) t.push_back(GemmTile{gi, a, b, groups[gi].seg_begin});
    }
    return t;
}

struct ProductPlan {
    int opA = 0, opB = 0;
    Layout out;
    std::vector<GemmTile> tiles;
    std::vector<GemmGroup> groups;
    std::vector<GemmSeg> segs;
    double flop = 0;     // 8*m*n*k summed over block pairs
    double bytes = 0;    // operand + result bytes per complex element size 1
    double unique = 0;   // elements of A, B and the result, each counted once
};

// product<N1,N2,nc>(m1, m2, T1, T2) (holstein/product.h:61-201).
// 'N' contracts the last nc legs of A and the first nc legs of B; 'T'/'C' contract the
// first nc legs of A / the last nc legs of B, 'C' conjugating and negating the kept
// legs' dirs.  Blocks pair when all contracted legs agree in qn and shape; pairs with the
// same output charge tuple become the K segments of one output group.  With a target
// layout, output offsets come from it and target blocks without contributions become
// zero groups (so the kernel writes every element of the target).
inline ProductPlan plan_product(const Layout& A, const Layout& B, int nc, char opA, char opB,
                                const Layout* target = nullptr) {
    ProductPlan P;
    P.opA = op_code(opA);
    P.opB = op_code(opB);
    const int n1 = A.rank, n2 = B.rank;
    KV_REQUIRE(nc >= 1 && nc <= n1 && nc <= n2, ERR_ARG, "bad contraction count");
    KV_REQUIRE(n1 + n2 - 2 * nc >= 1 && n1 + n2 - 2 * nc <= MAXR, ERR_ARG, "bad result rank");
    const int iax1 = (opA == 'N') ? n1 - nc : 0;
    const int iax2 = (opB == 'N') ? 0 : n2 - nc;
    const int k1b = (opA == 'N') ? 0 : nc, k1e = (opA == 'N') ? n1 - nc : n1;
    const int k2b = (opB == 'N') ? nc : 0, k2e = (opB == 'N') ? n2 : n2 - nc;
    const int fac1 = (opA == 'C') ? -1 : 1, fac2 = (opB == 'C') ? -1 : 1;
    for (int ax = 0; ax < nc; ++ax)
        if (A.dirs[iax1 + ax] * fac1 != -1 * B.dirs[iax2 + ax] * fac2)
            throw Error(ERR_DIRS, "Contracted legs' directions mismatch");
    Layout out;
    out.rank = n1 + n2 - 2 * nc;
    {
        int r = 0;
        for (int a = k1b; a < k1e; ++a) out.dirs[r++] = A.dirs[a] * fac1;
        for (int a = k2b; a < k2e; ++a) out.dirs[r++] = B.dirs[a] * fac2;
    }
    // index B blocks by contracted (qn, shape)
    std::map<std::vector<int>, std::vector<int>> bidx;
    for (int j = 0; j < (int)B.blocks.size(); ++j) {
        std::vector<int> key(2 * nc);
        for (int ax = 0; ax < nc; ++ax) {
            key[ax] = B.blocks[j].qn[iax2 + ax];
            key[nc + ax] = B.blocks[j].shape[iax2 + ax];
        }
        bidx[key].push_back(j);
    }
    struct Acc {
        Idx shape;
        std::vector<std::pair<int, int>> pairs;
    };
    std::map<std::vector<int>, Acc> groups;
    for (int i = 0; i < (int)A.blocks.size(); ++i) {
        std::vector<int> key(2 * nc);
        for (int ax = 0; ax < nc; ++ax) {
            key[ax] = A.blocks[i].qn[iax1 + ax];
            key[nc + ax] = A.blocks[i].shape[iax1 + ax];
        }
        auto it = bidx.find(key);
        if (it == bidx.end()) continue;
        for (int j : it->second) {
            std::vector<int> q(out.rank);
            Idx sh{};
            int r = 0;
            for (int a = k1b; a < k1e; ++a, ++r) {
                q[r] = A.blocks[i].qn[a];
                sh[r] = A.blocks[i].shape[a];
            }
            for (int a = k2b; a < k2e; ++a, ++r) {
                q[r] = B.blocks[j].qn[a];
                sh[r] = B.blocks[j].shape[a];
            }
            auto g = groups.find(q);
            if (g == groups.end()) {
                Acc acc;
                acc.shape = sh;
                acc.pairs.push_back({i, j});
                groups.emplace(q, std::move(acc));
            } else {
                KV_REQUIRE(qn_equal(g->second.shape, sh, out.rank), ERR_ARG,
                           "product: equal output charges with different shapes");
                g->second.pairs.push_back({i, j});
            }
        }
    }
    if (target) {
        KV_REQUIRE(target->rank == out.rank, ERR_INTERNAL, "target layout rank mismatch");
        for (int r = 0; r < out.rank; ++r)
            KV_REQUIRE(target->dirs[r] == out.dirs[r], ERR_INTERNAL, "target layout dirs mismatch");
        out.blocks = target->blocks;
        out.total = target->total;
    } else {
        for (auto& kvp : groups) {
            BlockDesc bd;
            for (int r = 0; r < out.rank; ++r) bd.qn[r] = kvp.first[r];
            bd.shape = kvp.second.shape;
            out.blocks.push_back(bd);
        }
        out.finalize();
    }
    const int nkept1 = k1e - k1b;
    std::vector<char> covered(out.blocks.size(), 0);
    for (auto& kvp : groups) {
        Idx q{};
        for (int r = 0; r < out.rank; ++r) q[r] = kvp.first[r];
        const int ob = out.find(q);
        KV_REQUIRE(ob >= 0, ERR_INTERNAL, "product output block missing from target layout");
        KV_REQUIRE(qn_equal(out.blocks[ob].shape, kvp.second.shape, out.rank), ERR_INTERNAL,
                   "product output shape differs from target layout");
        covered[ob] = 1;
        GemmGroup g{};
        g.c_off = out.blocks[ob].off;
        int64_t m = 1, n = 1;
        for (int r = 0; r < nkept1; ++r) m *= kvp.second.shape[r];
        for (int r = nkept1; r < out.rank; ++r) n *= kvp.second.shape[r];
        KV_REQUIRE(m < (1ll << 31) && n < (1ll << 31), ERR_ARG, "block too large");
        g.m = (int)m;
        g.n = (int)n;
        g.ldc = (int)n;
        g.seg_begin = (int)P.segs.size();
        g.seg_count = (int)kvp.second.pairs.size();
        for (auto& pr : kvp.second.pairs) {
            const BlockDesc& ba = A.blocks[pr.first];
            const BlockDesc& bb = B.blocks[pr.second];
            int64_t k = 1;
            for (int ax = 0; ax < nc; ++ax) k *= ba.shape[iax1 + ax];
            GemmSeg s{};
            s.a_off = ba.off;
            s.b_off = bb.off;
            s.k = (int)k;
            s.lda = (opA == 'N') ? (int)k : (int)m;
            s.ldb = (opB == 'N') ? (int)n : (int)k;
            P.segs.push_back(s);
            P.flop += 8.0 * (double)m * (double)n * (double)k;
            P.bytes += (double)(m * k + k * n);
        }
        P.bytes += (double)(m * n);
        P.groups.push_back(g);
    }
    P.unique = (double)A.total + (double)B.total;
    // zero groups for target blocks that receive nothing
    for (size_t ob = 0; ob < out.blocks.size(); ++ob) {
        if (covered[ob]) continue;
        GemmGroup g{};
        g.c_off = out.blocks[ob].off;
        const int last = out.blocks[ob].shape[out.rank - 1];
        g.n = last;
        g.m = (int)(out.blocks[ob].size / last);
        g.ldc = last;
        g.seg_begin = (int)P.segs.size();
        g.seg_count = 0;
        P.groups.push_back(g);
    }
    P.tiles = cut_tiles(P.groups, 0);
    P.out = std::move(out);
    P.unique += (double)P.out.total;
    return P;
}

// A product plan's K ranges cut into nch chunks per group: chunk c's groups write the partial
// result of the c-th part of their K range at c * out.total, to be summed in chunk order.
struct SplitK {
    int nch = 1;
    std::vector<GemmGroup> groups;
    std::vector<GemmSeg> segs;
    std::vector<GemmTile> tiles;  // config 0
};

// K chunks of a plan.  An output of few tiles leaves most of the 256 CUs idle while each
// workgroup walks its whole K range alone, 1.1 us per 8-deep stage (an environment update's
// last product at D = 128, 16 levels: 6 tiles, K = 2048, 286 us whole, 17 + 4 us cut in 32).  Chunks
// double while the workgroups stay under kSplitWgs and the deepest group keeps kSplitDepth per chunk.
// Plans that are cut keep the 64x64 tile; the largest of them gain least over their tuned tile uncut (one-site
// H_eff, us: 4 channels, D = 704, 121 tiles 689 -> 413, D = 1024, 256 tiles 1257 -> 1133, split BF16 396 -> 308; two
// channels, D = 768, two levels 756 -> 735).
constexpr int kSplitWgs = 512, kSplitDepth = 64, kSplitMax = 32;
inline int split_chunks(const ProductPlan& P) {
    int64_t kmax = 0;
    for (const auto& g : P.groups) {
        int64_t k = 0;
        for (int s = 0; s < g.seg_count; ++s) k += P.segs[g.seg_begin + s].k;
        kmax = std::max(kmax, k);
    }
    int n = 1;
    while (2 * n <= kSplitMax && (int64_t)P.tiles.size() * 2 * n <= kSplitWgs && kmax / (2 * n) >= kSplitDepth) n *= 2;
    return n;
}

inline SplitK split_k(const ProductPlan& P, int nch) {
    SplitK S;
    S.nch = nch;
    for (int c = 0; c < nch; ++c)
        for (const auto& g : P.groups) {
            int64_t K = 0;
            for (int s = 0; s < g.seg_count; ++s) K += P.segs[g.seg_begin + s].k;
            // chunk boundaries at multiples of 8, so that no stage of the kernel is cut short
            // where the segments allow it
            const int64_t per = ((K + nch - 1) / nch + 7) / 8 * 8;
            const int64_t lo = std::min(K, c * per), hi = std::min(K, lo + per);
            GemmGroup h = g;
            h.c_off = g.c_off + (int64_t)c * P.out.total;
            h.seg_begin = (int)S.segs.size();
            int64_t at = 0;
            for (int s = 0; s < g.seg_count; ++s) {
                const GemmSeg& sg = P.segs[g.seg_begin + s];
                const int64_t a = std::max(lo, at), b = std::min(hi, at + sg.k);
                if (a < b) {
                    const int64_t k0 = a - at;
                    GemmSeg t = sg;
                    t.a_off += P.opA == 0 ? k0 : k0 * sg.lda;
                    t.b_off += P.opB == 0 ? k0 * sg.ldb : k0;
                    t.k = (int)(b - a);
                    S.segs.push_back(t);
                }
                at += sg.k;
            }
            h.seg_count = (int)S.segs.size() - h.seg_begin;
            S.groups.push_back(h);
        }
    S.tiles = cut_tiles(S.groups, 0);
    return S;
}

struct WFoldPlan {
    Layout out;
    std::vector<WTask> tasks;
    std::vector<WTerm> terms;
    int maxP = 0;
    int64_t maxPQ = 0;  // largest task's P x Q
    double flop = 0;
    // host-side provenance for compose_wfold: per task (output block, s', wR), -1s for a
    // zero task; per term (input block, wL, s)
    std::vector<std::array<int, 3>> task_src, term_src;
};

// MPO fold (the env_mps_mpo family, holstein/product.h:203-477):
//   Y[pre, s', wR, post] = sum_{wL, s} W[s', wL, s, wR] X[pre, wL, s, post]
// where X legs p, p+1 pair with W legs 1 (wL) and 2 (s) on equal qn and shape.  W is
// tiny and sparse, so each nonzero W entry becomes a scaled slice term; every (s', wR)
// row of every output block is one task summing its terms.
inline WFoldPlan plan_wfold(const Layout& X, int p, const Layout& W, const double* Wd,
                            const Layout* target = nullptr) {
    WFoldPlan F;
    KV_REQUIRE(W.rank == 4, ERR_ARG, "MPO tensor must have rank 4");
    KV_REQUIRE(p >= 0 && p + 2 <= X.rank, ERR_ARG, "bad MPO fold position");
    Layout out;
    out.rank = X.rank;
    {
        int r = 0;
        for (int a = 0; a < p; ++a) out.dirs[r++] = X.dirs[a];
        out.dirs[r++] = W.dirs[0];
        out.dirs[r++] = W.dirs[3];
        for (int a = p + 2; a < X.rank; ++a) out.dirs[r++] = X.dirs[a];
    }
    std::map<std::vector<int>, std::vector<int>> widx;  // (wL qn, s qn, wL dim, s dim)
    for (int j = 0; j < (int)W.blocks.size(); ++j) {
        const auto& b = W.blocks[j];
        widx[{b.qn[1], b.qn[2], b.shape[1], b.shape[2]}].push_back(j);
    }
    struct Acc {
        Idx shape;
        std::vector<std::pair<int, int>> pairs;
    };
    std::map<std::vector<int>, Acc> groups;
    for (int i = 0; i < (int)X.blocks.size(); ++i) {
        const auto& xb = X.blocks[i];
        auto it = widx.find({xb.qn[p], xb.qn[p + 1], xb.shape[p], xb.shape[p + 1]});
        if (it == widx.end()) continue;
        for (int j : it->second) {
            const auto& wb = W.blocks[j];
            std::vector<int> q(out.rank);
            Idx sh{};
            int r = 0;
            for (int a = 0; a < p; ++a, ++r) {
                q[r] = xb.qn[a];
                sh[r] = xb.shape[a];
            }
            q[r] = wb.qn[0];
            sh[r++] = wb.shape[0];
            q[r] = wb.qn[3];
            sh[r++] = wb.shape[3];
            for (int a = p + 2; a < X.rank; ++a, ++r) {
                q[r] = xb.qn[a];
                sh[r] = xb.shape[a];
            }
            auto g = groups.find(q);
            if (g == groups.end()) {
                Acc acc;
                acc.shape = sh;
                acc.pairs.push_back({i, j});
                groups.emplace(q, std::move(acc));
            } else {
                KV_REQUIRE(qn_equal(g->second.shape, sh, out.rank), ERR_ARG,
                           "MPO fold: equal output charges with different shapes");
                g->second.pairs.push_back({i, j});
            }
        }
    }
    if (target) {
        out.blocks = target->blocks;
        out.total = target->total;
    } else {
        for (auto& kvp : groups) {
            BlockDesc bd;
            for (int r = 0; r < out.rank; ++r) bd.qn[r] = kvp.first[r];
            bd.shape = kvp.second.shape;
            out.blocks.push_back(bd);
        }
        out.finalize();
    }
    std::vector<char> covered(out.blocks.size(), 0);
    // nonzero entries of each W block by (s', wR) row, in the order (wL, s)
    struct Nz {
        int wl, s;
        double re, im;
    };
    struct Rows {
        std::vector<int> begin;
        std::vector<Nz> nz;
    };
    std::vector<Rows> wrows(W.blocks.size());
    auto rows_of = [&](int j) -> const Rows& {
        Rows& R = wrows[j];
        if (!R.begin.empty()) return R;
        const BlockDesc& wb = W.blocks[j];
        const int WR = wb.shape[3];
        const int64_t per = (int64_t)wb.shape[1] * wb.shape[2] * WR;
        R.begin.assign((size_t)wb.shape[0] * WR + 1, 0);
        const double* d = Wd + 2 * wb.off;
        for (int64_t e = 0; e < wb.size; ++e)
            if (d[2 * e] != 0.0 || d[2 * e + 1] != 0.0) R.begin[(e / per) * WR + e % WR + 1] += 1;
        for (size_t r = 1; r < R.begin.size(); ++r) R.begin[r] += R.begin[r - 1];
        R.nz.resize(R.begin.back());
        std::vector<int> at(R.begin.begin(), R.begin.end() - 1);
        for (int64_t e = 0; e < wb.size; ++e)
            if (d[2 * e] != 0.0 || d[2 * e + 1] != 0.0) {
                const int64_t in = e % per / WR;
                R.nz[at[(e / per) * WR + e % WR]++] = Nz{(int)(in / wb.shape[2]), (int)(in % wb.shape[2]), d[2 * e], d[2 * e + 1]};
            }
        return R;
    };
    for (auto& kvp : groups) {
        Idx q{};
        for (int r = 0; r < out.rank; ++r) q[r] = kvp.first[r];
        const int ob = out.find(q);
        KV_REQUIRE(ob >= 0, ERR_INTERNAL, "MPO fold output block missing from target");
        covered[ob] = 1;
        const BlockDesc& O = out.blocks[ob];
        int64_t Pd = 1, Qd = 1;
        for (int a = 0; a < p; ++a) Pd *= O.shape[a];
        for (int a = p + 2; a < out.rank; ++a) Qd *= O.shape[a];
        const int Sp = O.shape[p], WR = O.shape[p + 1];
        KV_REQUIRE(Pd < (1ll << 31) && Qd < (1ll << 31), ERR_ARG, "block too large");
        F.maxP = std::max<int>(F.maxP, (int)Pd);
        KV_REQUIRE(Pd * Qd < (1ll << 31), ERR_ARG, "MPO fold: block too large");
        F.maxPQ = std::max<int64_t>(F.maxPQ, Pd * Qd);
        for (int sp = 0; sp < Sp; ++sp)
            for (int wr = 0; wr < WR; ++wr) {
                WTask t{};
                t.out_base = O.off + ((int64_t)sp * WR + wr) * Qd;
                t.out_pstride = (int64_t)Sp * WR * Qd;
                t.P = (int)Pd;
                t.Q = (int)Qd;
                t.term_begin = (int)F.terms.size();
                for (auto& pr : kvp.second.pairs) {
                    const BlockDesc& xb = X.blocks[pr.first];
                    const int WL = xb.shape[p], S = xb.shape[p + 1];
                    const Rows& R = rows_of(pr.second);
                    const int row = sp * WR + wr;
                    for (int e = R.begin[row]; e < R.begin[row + 1]; ++e) {
                        const Nz& z = R.nz[e];
                        WTerm w{};
                        w.in_base = xb.off + ((int64_t)z.wl * S + z.s) * Qd;
                        w.in_pstride = (int64_t)WL * S * Qd;
                        w.re = z.re;
                        w.im = z.im;
                        F.terms.push_back(w);
                        F.term_src.push_back({pr.first, z.wl, z.s});
                        F.flop += 8.0 * (double)Pd * (double)Qd;
                    }
                }
                t.term_count = (int)F.terms.size() - t.term_begin;
                F.tasks.push_back(t);
                F.task_src.push_back({ob, sp, wr});
            }
    }
    for (size_t ob = 0; ob < out.blocks.size(); ++ob) {
        if (covered[ob]) continue;
        WTask t{};
        t.out_base = out.blocks[ob].off;
        t.out_pstride = 0;
        t.P = 1;
        KV_REQUIRE(out.blocks[ob].size < (1ll << 31), ERR_ARG, "block too large");
        t.Q = (int)out.blocks[ob].size;
        t.term_begin = (int)F.terms.size();
        t.term_count = 0;
        F.maxP = std::max(F.maxP, 1);
        F.maxPQ = std::max<int64_t>(F.maxPQ, t.Q);
        F.tasks.push_back(t);
        F.task_src.push_back({-1, -1, -1});
    }
    F.out = std::move(out);
    return F;
}

// The two folds of the two-site H_eff as one pass: F1 = plan_wfold(X, 1, W1) takes
// X[pre, wL, s1, s2, post] to Y[pre, s1', w1, s2, post] and F2 = plan_wfold(Y, 2, W2) takes
// Y to Z[pre, s1', s2', wR, post].  The composite reads X directly:
//   Z[pre, s1', s2', wR, post] = sum_{w1, s2} W2[s2', w1, s2, wR]
//                                  sum_{wL, s1} W1[s1', wL, s1, w1] X[pre, wL, s1, s2, post],
// one task per (F2 task, s1') over P = pre, Q = post, with a term per pair of nonzero W
// entries (weight W2 W1, X's slice of F1's term shifted to s2).  Z's layout is F2's.
// Only the two folds' own lists are built here: at 64 levels the composite has 49k tasks of
// 231k terms, which took 15 to 20 ms to list on the host and 10 MB to upload; a kernel expands
// them (wcompose_expand) in 9 us.
struct ComposePlan {
    std::vector<WComposeTask> tasks;   // one per F2 task
    std::vector<WComposeTerm> terms;   // one per F2 term
    int ntasks = 0;                    // composite tasks and term slots
    int64_t nterms = 0;
    int64_t maxPQ = 0;
    double flop = 0;
};

inline ComposePlan plan_compose(const WFoldPlan& F1, const WFoldPlan& F2, const Layout& Y) {
    KV_REQUIRE(F1.term_src.size() == F1.terms.size() && F2.term_src.size() == F2.terms.size() &&
                   F1.task_src.size() == F1.tasks.size() && F2.task_src.size() == F2.tasks.size(),
               ERR_INTERNAL, "plan_compose: plans without provenance");
    ComposePlan C;
    // F1's first task writing Y block yb (its tasks follow in the order s1', w1)
    std::vector<int> first(Y.blocks.size(), -1);
    for (size_t t = F1.tasks.size(); t-- > 0;)
        if (F1.task_src[t][0] >= 0) first[F1.task_src[t][0]] = (int)t;
    C.terms.reserve(F2.terms.size());
    for (size_t t2 = 0; t2 < F2.tasks.size(); ++t2) {
        const WTask& T2 = F2.tasks[t2];
        WComposeTask c{};
        c.out_base = T2.out_base;
        c.Q = T2.Q;
        c.task0 = C.ntasks;
        c.slot = C.nterms;
        c.term_begin = (int)C.terms.size();
        if (F2.task_src[t2][0] < 0) {  // an output block no term reaches: zeros
            c.out_pstride = T2.out_pstride;
            c.P = T2.P;
            c.S1 = 1;
        } else {
            const int S1 = F2.out.blocks[F2.task_src[t2][0]].shape[1];  // F2's pre is (pre, s1')
            KV_REQUIRE(S1 > 0 && T2.P % S1 == 0, ERR_INTERNAL, "plan_compose: pre does not end in s1'");
            c.out_pstride = (int64_t)S1 * T2.out_pstride;
            c.s1_stride = T2.out_pstride;
            c.P = T2.P / S1;
            c.S1 = S1;
            for (int k2 = T2.term_begin; k2 < T2.term_begin + T2.term_count; ++k2) {
                const auto& src = F2.term_src[k2];  // (Y block, w1, s2)
                WComposeTerm w{};
                w.shift = (int64_t)src[2] * T2.Q;
                w.re = F2.terms[k2].re;
                w.im = F2.terms[k2].im;
                w.f1_task = first[src[0]] < 0 ? -1 : first[src[0]] + src[1];
                w.f1_stride = Y.blocks[src[0]].shape[2];
                KV_REQUIRE(w.f1_task < 0 || F1.tasks[w.f1_task].P == c.P, ERR_INTERNAL,
                           "plan_compose: pre extents differ");
                C.terms.push_back(w);
            }
            c.term_count = (int)C.terms.size() - c.term_begin;
            for (int s1 = 0; s1 < S1; ++s1) {
                int nt = 0;
                for (int k = c.term_begin; k < c.term_begin + c.term_count; ++k)
                    if (C.terms[k].f1_task >= 0)
                        nt += F1.tasks[C.terms[k].f1_task + s1 * C.terms[k].f1_stride].term_count;
                c.maxt = std::max(c.maxt, nt);
                C.flop += 8.0 * nt * (double)c.P * (double)c.Q;
            }
        }
        C.ntasks += c.S1;
        C.nterms += (int64_t)c.S1 * c.maxt;
        KV_REQUIRE(C.nterms < (1ll << 31), ERR_ARG, "MPO fold: too many terms");
        C.maxPQ = std::max<int64_t>(C.maxPQ, (int64_t)c.P * c.Q);
        C.tasks.push_back(c);
    }
    return C;
}

// The composite's lists, expanded on the host: for plans checked without a GPU (the engine expands them on
// the device).
inline WFoldPlan compose_wfold(const WFoldPlan& F1, const WFoldPlan& F2, const Layout& Y) {
    const ComposePlan C = plan_compose(F1, F2, Y);
    WFoldPlan W;
    W.out = F2.out;
    W.tasks.resize(C.ntasks);
    W.terms.resize(C.nterms);
    W.maxPQ = C.maxPQ;
    W.flop = C.flop;
    for (const auto& c : C.tasks) {
        W.maxP = std::max(W.maxP, c.P);
        for (int s1 = 0; s1 < c.S1; ++s1)
            wcompose_expand(c, s1, C.terms.data(), F1.tasks.data(), F1.terms.data(), W.tasks.data(), W.terms.data());
    }
    return W;
}

struct PermPlan {
    Layout out;
    std::vector<PermTask> tasks;
    int64_t maxsize = 0;
};

// Leg permutation out-leg r = in-leg axes[r] (holstein/tensor.h:244-260).
inline PermPlan plan_perm(const Layout& X, const Idx& axes) {
    PermPlan P;
    P.out.rank = X.rank;
    for (int r = 0; r < X.rank; ++r) P.out.dirs[r] = X.dirs[axes[r]];
    for (const auto& b : X.blocks) {
        BlockDesc o;
        for (int r = 0; r < X.rank; ++r) {
            o.qn[r] = b.qn[axes[r]];
            o.shape[r] = b.shape[axes[r]];
        }
        P.out.blocks.push_back(o);
    }
    P.out.finalize();
    for (const auto& b : X.blocks) {
        Idx q{};
        for (int r = 0; r < X.rank; ++r) q[r] = b.qn[axes[r]];
        const int ob = P.out.find(q);
        PermTask t{};
        t.in_off = b.off;
        t.out_off = P.out.blocks[ob].off;
        t.size = b.size;
        t.rank = X.rank;
        int64_t istr[MAXR];
        int64_t s = 1;
        for (int r = X.rank - 1; r >= 0; --r) {
            istr[r] = s;
            s *= b.shape[r];
        }
        for (int r = 0; r < X.rank; ++r) {
            t.oshape[r] = b.shape[axes[r]];
            t.istride[r] = istr[axes[r]];
        }
        P.maxsize = std::max(P.maxsize, b.size);
        P.tasks.push_back(t);
    }
    return P;
}

// Host-side permutation of a small tensor (used for MPO tensors, which live on the host).
inline void host_perm(const Layout& X, const double* d, const Idx& axes, Layout& out,
                      std::vector<double>& od) {
    PermPlan P = plan_perm(X, axes);
    out = P.out;
    od.assign(2 * (size_t)out.total, 0.0);
    for (const auto& t : P.tasks) {
        for (int64_t e = 0; e < t.size; ++e) {
            int64_t rem = e, src = 0;
            for (int r = t.rank - 1; r >= 0; --r) {
                const int64_t idx = rem % t.oshape[r];
                rem /= t.oshape[r];
                src += idx * t.istride[r];
            }
            od[2 * (t.out_off + e)] = d[2 * (t.in_off + src)];
            od[2 * (t.out_off + e) + 1] = d[2 * (t.in_off + src) + 1];
        }
    }
}

// Effective-Hamiltonian plan.  nsite = 2: apply_double (holstein/product.h:478-486) as
//   T1 = L.x (product<3,4,1>), T2 = fold W1 at legs (1,2), T3 = fold W2 at legs (2,3),
//   y = T3.R^T (product<5,3,2>, N/T);
// nsite = 1: apply_single (:547-553) T1 = L.x, T2 = fold W at (1,2), y = T2.R^T;
// nsite = 0: apply_zero (:540-545) T1 = L.C, y = T1.R^T.
// The vector layout xl is the closure of x's blocks under H_eff, so every Krylov vector
// shares one slab layout.
struct HeffStructure {
    int nsite = 2;
    Layout xl;
    ProductPlan s1, s4;
    WFoldPlan s2, s3;
    WFoldPlan s23;  // two sites, where asked for: both folds as one pass, expanded on the host
    double flop = 0;
};

inline HeffStructure plan_heff(int nsite, const Layout& L, const Layout* W1, const double* W1d,
                               const Layout* W2, const double* W2d, const Layout& R,
                               const Layout& x, bool composite = true) {
    KV_REQUIRE(nsite >= 0 && nsite <= 2, ERR_ARG, "nsite must be 0, 1 or 2");
    KV_REQUIRE(x.rank == nsite + 2, ERR_ARG, "x rank does not match nsite");
    HeffStructure H;
    H.nsite = nsite;
    Layout cur = x;
    for (int it = 0; it < 16; ++it) {
        H.s1 = plan_product(L, cur, 1, 'N', 'N');
        const Layout* t = &H.s1.out;
        if (nsite >= 1) {
            H.s2 = plan_wfold(*t, 1, *W1, W1d);
            t = &H.s2.out;
        }
        if (nsite == 2) {
            H.s3 = plan_wfold(*t, 2, *W2, W2d);
            t = &H.s3.out;
        }
        ProductPlan probe = plan_product(*t, R, 2, 'N', 'T');
        Layout u = union_layout(cur, probe.out);
        if (same_layout(u, cur)) break;
        KV_REQUIRE(it < 15, ERR_INTERNAL, "H_eff block closure did not converge");
        cur = u;
    }
    const Layout* t = nsite == 2 ? &H.s3.out : (nsite == 1 ? &H.s2.out : &H.s1.out);
    H.s4 = plan_product(*t, R, 2, 'N', 'T', &cur);
    H.xl = cur;
    if (nsite == 2 && composite) H.s23 = compose_wfold(H.s2, H.s3, H.s2.out);
    H.flop = H.s1.flop + H.s2.flop + H.s3.flop + H.s4.flop;
    return H;
}

// Environment update env_sweep (holstein/product.h:488-521).  L2R:
//   lm = env.ket (product<3,3,1>), lmo = fold W at (1,2), out = bra^dag.lmo (product<3,4,2>, C/N).
// R2L applies the same after transposing bra/ket by (2,1,0) and W by (0,3,2,1); the
// caller does those permutations.
struct EnvStructure {
    ProductPlan s1, s3;
    WFoldPlan s2;
    double flop = 0;
};

inline EnvStructure plan_env_l2r(const Layout& env, const Layout& bra, const Layout& W,
                                 const double* Wd, const Layout& ket) {
    EnvStructure E;
    E.s1 = plan_product(env, ket, 1, 'N', 'N');
    E.s2 = plan_wfold(E.s1.out, 1, W, Wd);
    E.s3 = plan_product(bra, E.s2.out, 2, 'C', 'N');
    E.flop = E.s1.flop + E.s2.flop + E.s3.flop;
    return E;
}

}  // namespace kv
