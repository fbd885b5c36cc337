// Executors of the contraction plans: block-sparse product, MPO fold, transposes, the
// effective-Hamiltonian matvec and the environment update, all on the context stream.
#pragma once

#include <cstdio>
#include <cstdlib>
#include <memory>
#include <type_traits>
#include <vector>

#include "plan.h"
#include "tensor.h"

namespace kv {

// PREC_BF16X3: FP32 storage, GEMMs as split-BF16 products with FP32 accumulation
enum Prec { PREC_F64 = 0, PREC_F32 = 1, PREC_BF16X3 = 2 };

// Times of the contraction launches, from the device's wall clock: a launch is marked as it
// starts and ends where the next mark stands (kv_kernels.h); resolved after the host has
// synchronised the stream anyway.  Events around each launch were packets of their own between
// the kernels and several host calls a launch: a third of a step of small tensors.
class MarkLog {
  public:
    explicit MarkLog(Device& dev) : dev_(dev) {
        int khz = 0;
        KV_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev.id));
        ms_per_tick_ = 1.0 / (double)(khz > 0 ? khz : 100000);
    }
    MarkLog(const MarkLog&) = delete;
    MarkLog& operator=(const MarkLog&) = delete;
    ~MarkLog() {
        dev_.mark_chunks.insert(dev_.mark_chunks.end(), chunks_.begin(), chunks_.end());
    }
    // The mark of a launch of this kind: 0 gemm (FP64 operands), 1 wfold, 2 gemm (FP32 operands);
    // bytes: operands and result once each.
    Mark* begin(int kind, double flop, double bytes) {
        Mark* m = slot();
        pending_.push_back({m, flop, bytes, kind});
        return m;
    }
    // The mark that ends the last launch (nothing, where none has begun since the last end).
    Mark* end() {
        if (pending_.empty() || pending_.back().kind < 0) return nullptr;
        Mark* m = slot();
        pending_.push_back({m, 0.0, 0.0, -1});
        return m;
    }
    size_t size() const { return pending_.size(); }
    // forgets the records from the n-th on (launches that found their iteration stopped)
    void drop(size_t n) { pending_.resize(n); }
    // call only after the stream has been synchronised
    void resolve(KernelStats& st) {
        for (size_t i = 0; i + 1 < pending_.size(); ++i) {
            const Rec& r = pending_[i];
            if (r.kind < 0) continue;
            const double ms = ms_per_tick_ * (double)(*pending_[i + 1].at - *r.at);
            if (r.kind == 1) {
                st.wfold_ms += ms;
                st.wfold_flop += r.flop;
                st.wfold_launches += 1;
                continue;
            }
            st.gemm_ms += ms;
            st.gemm_flop += r.flop;
            st.gemm_bytes += r.bytes;
            st.gemm_launches += 1;
            if (r.kind == 2) {
                st.gemm32_ms += ms;
                st.gemm32_flop += r.flop;
                st.gemm32_bytes += r.bytes;
                st.gemm32_launches += 1;
            }
        }
        pending_.clear();
        used_ = 0;
    }

  private:
    struct Rec {
        Mark* at;
        double flop, bytes;
        int kind;  // -1: an end
    };
    static constexpr size_t kChunk = Device::kMarkChunk;
    Mark* slot() {
        if (used_ == chunks_.size() * kChunk) chunks_.push_back(dev_.mark_chunk());
        Mark* m = chunks_[used_ / kChunk] + used_ % kChunk;
        ++used_;
        return m;
    }
    Device& dev_;
    std::vector<Mark*> chunks_;
    size_t used_ = 0;
    std::vector<Rec> pending_;
    double ms_per_tick_ = 1e-5;
};

// Shape class of a product plan for the tile autotuner: log2 buckets of the m, n and total
// k of its largest group.
inline uint64_t gemm_shape_key(const ProductPlan& p, int prec) {
    int64_t best = -1;
    int bm = 0, bn = 0, bk = 0;
    for (const auto& g : p.groups) {
        int64_t k = 0;
        for (int s = 0; s < g.seg_count; ++s) k += p.segs[g.seg_begin + s].k;
        const int64_t w = (int64_t)g.m * g.n * std::max<int64_t>(k, 1);
        if (w > best) {
            best = w;
            bm = g.m;
            bn = g.n;
            bk = (int)std::min<int64_t>(k, 1 << 30);
        }
    }
    auto lg = [](int v) {
        int l = 0;
        while ((1 << (l + 1)) <= v && l < 20) ++l;
        return l;
    };
    return ((uint64_t)prec << 40) | ((uint64_t)p.opA << 36) | ((uint64_t)p.opB << 32) |
           ((uint64_t)lg(bm) << 20) | ((uint64_t)lg(bn) << 10) | (uint64_t)lg(bk);
}

struct DevProduct {
    ProductPlan p;
    const GemmGroup* groups = nullptr;  // in the lists the plan was staged with
    const GemmSeg* segs = nullptr;
    DevBuf tiles[kNumGemmConfigs];  // other configs' tiles than 0, cut on first use
    const GemmTile* tp[kNumGemmConfigs] = {nullptr};
    int ntiles[kNumGemmConfigs] = {0};
    bool cut[kNumGemmConfigs] = {false};
    int nch = 1;   // K chunks (split_chunks): above 1 the lists are split_k's
    DevBuf part;   // and the chunks' partial results go here, one after the other
    size_t off[3] = {0, 0, 0};
    // the plan's groups, segments and config 0's tiles into L; bind() after L's commit
    void stage(Device& dev, ProductPlan plan, StagedLists& L) {
        p = std::move(plan);
        nch = split_chunks(p);
        auto put = [&](const auto& lists) {
            off[0] = L.stage(lists.groups);
            off[1] = L.stage(lists.segs);
            off[2] = L.stage(lists.tiles);
            ntiles[0] = (int)lists.tiles.size();
        };
        if (nch > 1) {
            part = DevBuf(dev.pool.get(), (size_t)nch * p.out.total * sizeof(double2));
            put(split_k(p, nch));
        } else {
            put(p);
        }
        cut[0] = true;
    }
    void bind(const StagedLists& L) {
        groups = L.at<GemmGroup>(off[0]);
        segs = L.at<GemmSeg>(off[1]);
        tp[0] = L.at<GemmTile>(off[2]);
    }
    void ensure_tiles(Device& dev, int cfg) {
        if (cut[cfg]) return;
        std::vector<GemmTile> t = cut_tiles(nch > 1 ? split_k(p, nch).groups : p.groups, cfg);
        tiles[cfg] = upload_vec(dev, t);
        tp[cfg] = tiles[cfg].as<GemmTile>();
        ntiles[cfg] = (int)t.size();
        cut[cfg] = true;
    }
    template <class T2>
    void launch(Device& dev, int cfg, const T2* A, const T2* B, T2* C, double ar, double ai,
                const int* stop = nullptr, Mark* mark = nullptr) {
        ensure_tiles(dev, cfg);
        launch_gemm<T2>(dev.stream, p.opA, p.opB, A, B, nch > 1 ? part.as<T2>() : C, tp[cfg], ntiles[cfg],
                        groups, segs, ar, ai, cfg, stop, mark);
        if (nch > 1) launch_sum_parts<T2>(dev.stream, part.as<T2>(), nch, p.out.total, C, stop);
    }
    // Ends the log's open record: the launches that time the tiles are no part of it.
    static void close(Device& dev, MarkLog* log) {
        if (Mark* done = log ? log->end() : nullptr) launch_mark(dev.stream, done);
    }
    // Tile config for this plan: cached per shape class; on a first encounter every config
    // built for the op pair runs twice on the real operands and the fastest is kept.
    template <class T2>
    int choose(Device& dev, const T2* A, const T2* B, T2* C, double ar, double ai, MarkLog* log) {
        if (!dev.autotune || p.flop < 1e8 || nch > 1) return 0;
        const uint64_t key = gemm_shape_key(p, sizeof(T2) == sizeof(double2) ? 0 : 1);
        auto it = dev.gemm_tuned.find(key);
        if (it != dev.gemm_tuned.end()) return it->second;
        close(dev, log);
        EventTimer ev;
        int best = 0;
        float best_ms = 1e30f;
        const char* vb = std::getenv("KV_VERBOSE");
        const bool verbose = vb && vb[0] == '1';
        char line[512];
        int len = std::snprintf(line, sizeof line, "[kv] autotune %s op%d%d %.3g GFLOP:",
                                sizeof(T2) == sizeof(double2) ? "f64" : "f32", p.opA, p.opB,
                                p.flop * 1e-9);
        for (int cfg = 0; cfg < kNumGemmConfigs; ++cfg) {
            if (!gemm_config_supports(cfg, p.opA, p.opB, sizeof(T2) == sizeof(double2))) continue;
            launch<T2>(dev, cfg, A, B, C, ar, ai);
            ev.start(dev.stream);
            launch<T2>(dev, cfg, A, B, C, ar, ai);
            ev.stop(dev.stream);
            const float ms = ev.ms();
            if (verbose && len < (int)sizeof line - 40)
                len += std::snprintf(line + len, sizeof line - len, " %dx%dx%d=%.3fms",
                                     kGemmConfigs[cfg].bm, kGemmConfigs[cfg].bn,
                                     kGemmConfigs[cfg].bk, ms);
            if (ms < best_ms) {
                best_ms = ms;
                best = cfg;
            }
        }
        if (verbose) std::fprintf(stderr, "%s -> %d\n", line, best);
        dev.gemm_tuned[key] = best;
        return best;
    }
    void launch_split(Device& dev, int cfg, const float2* A, const float2* B, float2* C, double ar,
                      double ai, const int* stop = nullptr, Mark* mark = nullptr) {
        ensure_tiles(dev, cfg);
        launch_gemm_bf16x3(dev.stream, p.opA, p.opB, A, B, nch > 1 ? part.as<float2>() : C, tp[cfg], ntiles[cfg],
                           groups, segs, ar, ai, cfg, stop, mark);
        if (nch > 1) launch_sum_parts<float2>(dev.stream, part.as<float2>(), nch, p.out.total, C, stop);
    }
    // Split-BF16 tile (64x64 or 128x128): KV_SPLIT_TILE's, also for a plan cut into K chunks, else
    // timed once per shape class like choose().
    int choose_split(Device& dev, const float2* A, const float2* B, float2* C, double ar, double ai, MarkLog* log) {
        if (const char* t = std::getenv("KV_SPLIT_TILE")) return std::atoi(t) == 128 ? 4 : 0;
        if (!dev.autotune || p.flop < 1e8 || nch > 1) return 0;
        const uint64_t key = gemm_shape_key(p, 2);
        auto it = dev.gemm_tuned.find(key);
        if (it != dev.gemm_tuned.end()) return it->second;
        close(dev, log);
        EventTimer ev;
        int best = 0;
        float best_ms = 1e30f;
        for (int cfg : {0, 4}) {
            launch_split(dev, cfg, A, B, C, ar, ai);
            ev.start(dev.stream);
            launch_split(dev, cfg, A, B, C, ar, ai);
            ev.stop(dev.stream);
            const float ms = ev.ms();
            if (ms < best_ms) {
                best_ms = ms;
                best = cfg;
            }
        }
        dev.gemm_tuned[key] = best;
        return best;
    }
    template <class T2>
    void run(Device& dev, const T2* A, const T2* B, T2* C, double alpha_re = 1.0,
             double alpha_im = 0.0, MarkLog* log = nullptr, bool split = false, const int* stop = nullptr) {
        int cfg = 0;
        if constexpr (std::is_same<T2, float2>::value) {
            cfg = split ? choose_split(dev, A, B, C, alpha_re, alpha_im, log)
                        : choose<T2>(dev, A, B, C, alpha_re, alpha_im, log);
        } else {
            cfg = choose<T2>(dev, A, B, C, alpha_re, alpha_im, log);
        }
        Mark* mark = nullptr;
        if (log && !p.tiles.empty())
            mark = log->begin(sizeof(T2) == sizeof(float2) ? 2 : 0, p.flop, p.unique * (double)sizeof(T2));
        if constexpr (std::is_same<T2, float2>::value) {
            if (split)
                launch_split(dev, cfg, A, B, C, alpha_re, alpha_im, stop, mark);
            else
                launch<T2>(dev, cfg, A, B, C, alpha_re, alpha_im, stop, mark);
        } else {
            KV_REQUIRE(!split, ERR_INTERNAL, "split-BF16 GEMM takes FP32 operands");
            launch<T2>(dev, cfg, A, B, C, alpha_re, alpha_im, stop, mark);
        }
    }
};

struct DevWFold {
    WFoldPlan p;
    const WTask* tasks = nullptr;  // in the lists the plan was staged with
    const WTerm* terms = nullptr;
    size_t off[2] = {0, 0};
    void stage(WFoldPlan plan, StagedLists& L) {
        p = std::move(plan);
        off[0] = L.stage(p.tasks);
        off[1] = L.stage(p.terms);
    }
    void bind(const StagedLists& L) {
        tasks = L.at<WTask>(off[0]);
        terms = L.at<WTerm>(off[1]);
    }
    template <class T2>
    void run(Device& dev, const T2* in, T2* out, MarkLog* log = nullptr, const int* stop = nullptr) const {
        Mark* mark = log && !p.tasks.empty() ? log->begin(1, p.flop, 0.0) : nullptr;
        launch_wfold<T2>(dev.stream, in, out, tasks, (int)p.tasks.size(), terms, p.maxPQ, stop, mark);
    }
};

// The two folds of a two-site H_eff as one pass, its tasks expanded on the device.
struct DevCompose {
    int ntasks = 0;
    int64_t maxPQ = 0;
    double flop = 0;
    DevBuf tasks, terms;
    int ntasks2 = 0;
    size_t off[2] = {0, 0};
    void stage(Device& dev, const DevWFold& f1, const DevWFold& f2, StagedLists& L) {
        const ComposePlan C = plan_compose(f1.p, f2.p, f1.p.out);
        ntasks = C.ntasks;
        ntasks2 = (int)C.tasks.size();
        maxPQ = C.maxPQ;
        flop = C.flop;
        tasks = DevBuf(dev.pool.get(), (size_t)C.ntasks * sizeof(WTask));
        terms = DevBuf(dev.pool.get(), (size_t)C.nterms * sizeof(WTerm));
        off[0] = L.stage(C.tasks);
        off[1] = L.stage(C.terms);
    }
    // after L's commit and f1's bind
    void expand(Device& dev, const DevWFold& f1, const StagedLists& L) {
        launch_wcompose(dev.stream, L.at<WComposeTask>(off[0]), ntasks2, L.at<WComposeTerm>(off[1]), f1.tasks,
                        f1.terms, tasks.as<WTask>(), terms.as<WTerm>());
    }
    template <class T2>
    void run(Device& dev, const T2* in, T2* out, MarkLog* log, const int* stop) const {
        Mark* mark = log && ntasks > 0 ? log->begin(1, flop, 0.0) : nullptr;
        launch_wfold<T2>(dev.stream, in, out, tasks.as<WTask>(), ntasks, terms.as<WTerm>(), maxPQ, stop, mark);
    }
};

// product<N1,N2,nc>(m1, m2, T1, T2) on the device, FP64 (holstein/product.h:61-201).
inline std::unique_ptr<Tensor> product(const std::shared_ptr<Device>& dev, const Tensor& A,
                                       const Tensor& B, int nc, char opA, char opB) {
    DevProduct dp;
    StagedLists L;
    dp.stage(*dev, plan_product(A.lay, B.lay, nc, opA, opB), L);
    L.commit(*dev);
    dp.bind(L);
    auto C = Tensor::create(dev, dp.p.out, false);
    dp.run<double2>(*dev, A.d(), B.d(), C->d());
    return C;
}

// transpose(t, axes) on the device (holstein/tensor.h:244-260).
inline std::unique_ptr<Tensor> transpose(const std::shared_ptr<Device>& dev, const Tensor& X,
                                         const Idx& axes) {
    PermPlan P = plan_perm(X.lay, axes);
    auto Y = Tensor::create(dev, P.out, false);
    DevBuf tasks = upload_vec(*dev, P.tasks);
    launch_perm<double2>(dev->stream, X.d(), Y->d(), tasks.as<PermTask>(), (int)P.tasks.size(),
                         P.maxsize);
    return Y;
}

// Copy X into the (larger) layout `to`, zero elsewhere.
inline std::unique_ptr<Tensor> relayout(const std::shared_ptr<Device>& dev, const Tensor& X,
                                        const Layout& to) {
    if (same_layout(X.lay, to)) return X.clone();
    auto Y = Tensor::create(dev, to, true);
    std::vector<Copy2D> cps;
    int maxrows = 1;
    for (const auto& b : X.lay.blocks) {
        const int ob = to.find(b.qn);
        KV_REQUIRE(ob >= 0 && qn_equal(to.blocks[ob].shape, b.shape, to.rank), ERR_INTERNAL,
                   "relayout: block missing from target layout");
        const int last = b.shape[X.lay.rank - 1];
        Copy2D c{};
        c.src_off = b.off;
        c.dst_off = to.blocks[ob].off;
        c.rows = (int)(b.size / last);
        c.cols = last;
        c.src_ld = last;
        c.dst_ld = last;
        maxrows = std::max(maxrows, c.rows);
        cps.push_back(c);
    }
    if (!cps.empty()) {
        DevBuf d = upload_vec(*dev, cps);
        launch_copy2d<double2>(dev->stream, X.d(), Y->d(), d.as<Copy2D>(), (int)cps.size(),
                               maxrows, nullptr);
    }
    return Y;
}

// y + alpha x over the union of both tensors' blocks (holstein/tensor.h:173-186 appends a
// block with a new (shape, qn) and axpys into an equal one).
inline std::unique_ptr<Tensor> axpy(const std::shared_ptr<Device>& dev, const Tensor& X,
                                    const Tensor& Y, double2 alpha) {
    KV_REQUIRE(X.lay.rank == Y.lay.rank, ERR_ARG, "axpy: rank mismatch");
    for (int a = 0; a < X.lay.rank; ++a)
        KV_REQUIRE(X.lay.dirs[a] == Y.lay.dirs[a], ERR_DIRS, "axpy: leg directions differ");
    const Layout U = union_layout(X.lay, Y.lay);
    auto Xu = relayout(dev, X, U);
    auto out = relayout(dev, Y, U);
    launch_zaxpby(dev->stream, out->d(), Xu->d(), out->d(), alpha, make_double2(1.0, 0.0),
                  U.total);
    dev->sync();
    return out;
}

// Effective Hamiltonian on one bond / site, built once per Lanczos call
// (apply_double / apply_single / apply_zero, holstein/product.h:478-553).
struct Heff {
    std::shared_ptr<Device> dev;
    HeffStructure S;
    Prec prec = PREC_F64;
    StagedLists lists;
    DevProduct s1, s4;
    // the MPO folds; two sites in FP32 / split-BF16 also both folds as one pass (s23)
    DevWFold s2, s3;
    DevCompose s23;
    const Tensor* L = nullptr;
    const Tensor* R = nullptr;
    DevBuf L32, R32, x32, y32, t1, t2, t3;

    void build(const std::shared_ptr<Device>& d, int nsite, const Tensor& Lt, Tensor* W1,
               Tensor* W2, const Tensor& Rt, const Layout& x, Prec p) {
        dev = d;
        prec = p;
        L = &Lt;
        R = &Rt;
        const double* w1d = W1 ? W1->host_data().data() : nullptr;
        const double* w2d = W2 ? W2->host_data().data() : nullptr;
        S = plan_heff(nsite, Lt.lay, W1 ? &W1->lay : nullptr, w1d, W2 ? &W2->lay : nullptr, w2d,
                      Rt.lay, x, false);
        const bool one_pass = nsite == 2 && p != PREC_F64;
        s1.stage(*dev, S.s1, lists);
        if (nsite >= 1) s2.stage(S.s2, lists);
        if (nsite == 2) s3.stage(S.s3, lists);
        if (one_pass) s23.stage(*dev, s2, s3, lists);
        s4.stage(*dev, S.s4, lists);
        lists.commit(*dev);  // one upload for the launches of every stage
        s1.bind(lists);
        if (nsite >= 1) s2.bind(lists);
        if (nsite == 2) s3.bind(lists);
        if (one_pass) s23.expand(*dev, s2, lists);
        s4.bind(lists);
        // intermediates sized for FP64 so either precision can run through them
        const size_t es = sizeof(double2);
        t1 = DevBuf(dev->pool.get(), (size_t)S.s1.out.total * es);
        if (nsite >= 1) t2 = DevBuf(dev->pool.get(), (size_t)S.s2.out.total * es);
        if (nsite == 2) t3 = DevBuf(dev->pool.get(), (size_t)S.s3.out.total * es);
        if (p != PREC_F64) {
            L32 = DevBuf(dev->pool.get(), (size_t)Lt.lay.total * sizeof(float2));
            R32 = DevBuf(dev->pool.get(), (size_t)Rt.lay.total * sizeof(float2));
            x32 = DevBuf(dev->pool.get(), (size_t)S.xl.total * sizeof(float2));
            y32 = DevBuf(dev->pool.get(), (size_t)S.xl.total * sizeof(float2));
            launch_f64_to_f32(dev->stream, Lt.d(), L32.as<float2>(), Lt.lay.total);
            launch_f64_to_f32(dev->stream, Rt.d(), R32.as<float2>(), Rt.lay.total);
        }
    }
    const Layout& layout() const { return S.xl; }
    double flop() const { return S.flop; }

    template <class T2>
    void chain(const T2* Ld, const T2* Rd, const T2* x, T2* y, double alpha, MarkLog* log,
               bool split = false, const int* stop = nullptr) {
        s1.run<T2>(*dev, Ld, x, t1.as<T2>(), 1.0, 0.0, log, split, stop);
        const T2* last = t1.as<T2>();
        // FP64 keeps the two folds one after the other (the reference's order of sums);
        // the FP32 operands take the one-pass composite, which saves a pass over the
        // intermediate at the cost of a different rounding order
        const bool one_pass = S.nsite == 2 && !std::is_same<T2, double2>::value;
        if (one_pass) {
            s23.run<T2>(*dev, last, t3.as<T2>(), log, stop);
            last = t3.as<T2>();
        } else {
            if (S.nsite >= 1) {
                s2.run<T2>(*dev, last, t2.as<T2>(), log, stop);
                last = t2.as<T2>();
            }
            if (S.nsite == 2) {
                s3.run<T2>(*dev, last, t3.as<T2>(), log, stop);
                last = t3.as<T2>();
            }
        }
        s4.run<T2>(*dev, last, Rd, y, alpha, 0.0, log, split, stop);
    }
    // y = alpha * H_eff x, x and y FP64 slabs in layout() order; force64 runs the
    // contractions in FP64 whatever the plan's precision; stop: see kv_kernels.h.  The caller marks
    // the end of the last launch (log->end())
    void apply(const double2* x, double2* y, double alpha, MarkLog* log = nullptr,
               bool force64 = false, const int* stop = nullptr) {
        if (prec == PREC_F64 || force64) {
            chain<double2>(L->d(), R->d(), x, y, alpha, log, false, stop);
        } else {
            launch_f64_to_f32(dev->stream, x, x32.as<float2>(), S.xl.total, stop);
            chain<float2>(L32.as<float2>(), R32.as<float2>(), x32.as<float2>(), y32.as<float2>(),
                          1.0, log, prec == PREC_BF16X3, stop);
            launch_f32_to_f64(dev->stream, y32.as<float2>(), y, alpha, S.xl.total, stop, log ? log->end() : nullptr);
        }
    }
};

// env_sweep (holstein/product.h:488-521): L2R  L' = bra^dag . (L . ket . W);
// R2L: the same after transposing bra/ket (2,1,0) and W (0,3,2,1).  One upload carries the lists
// of every launch.  Without `wait` the result is ready in stream order.
inline std::unique_ptr<Tensor> env_update(const std::shared_ptr<Device>& dev, const Tensor& env,
                                          const Tensor* bra, Tensor& W, const Tensor& ket,
                                          bool l2r, Prec prec, MarkLog* log = nullptr,
                                          double* flop = nullptr, bool wait = true) {
    std::unique_ptr<Tensor> kt, bt;
    const Tensor* k = &ket;
    const Tensor* b = bra ? bra : &ket;
    Layout wl;
    std::vector<double> wt;
    const Layout* wlay = &W.lay;
    const double* wd = W.host_data().data();
    StagedLists L;
    PermPlan pk, pb;
    size_t pk_off = 0, pb_off = 0;
    if (!l2r) {
        const Idx ax{2, 1, 0, 0, 0, 0};
        pk = plan_perm(ket.lay, ax);
        pk_off = L.stage(pk.tasks);
        kt = Tensor::create(dev, pk.out, false);
        k = kt.get();
        if (bra) {
            pb = plan_perm(bra->lay, ax);
            pb_off = L.stage(pb.tasks);
            bt = Tensor::create(dev, pb.out, false);
            b = bt.get();
        } else {
            b = k;
        }
        host_perm(W.lay, wd, Idx{0, 3, 2, 1, 0, 0}, wl, wt);
        wlay = &wl;
        wd = wt.data();
    }
    EnvStructure E = plan_env_l2r(env.lay, b->lay, *wlay, wd, k->lay);
    if (flop) *flop += E.flop;
    DevProduct s1, s3;
    DevWFold s2;
    const size_t n1 = (size_t)E.s1.out.total, n2 = (size_t)E.s2.out.total;
    const int64_t n3 = E.s3.out.total;
    auto out = Tensor::create(dev, E.s3.out, false);
    s1.stage(*dev, std::move(E.s1), L);
    s2.stage(std::move(E.s2), L);
    s3.stage(*dev, std::move(E.s3), L);
    L.commit(*dev);
    s1.bind(L);
    s2.bind(L);
    s3.bind(L);
    if (kt)
        launch_perm<double2>(dev->stream, ket.d(), kt->d(), L.at<PermTask>(pk_off), (int)pk.tasks.size(), pk.maxsize);
    if (bt)
        launch_perm<double2>(dev->stream, bra->d(), bt->d(), L.at<PermTask>(pb_off), (int)pb.tasks.size(),
                             pb.maxsize);
    if (prec == PREC_F64) {
        DevBuf t1(dev->pool.get(), n1 * sizeof(double2));
        DevBuf t2(dev->pool.get(), n2 * sizeof(double2));
        s1.run<double2>(*dev, env.d(), k->d(), t1.as<double2>(), 1.0, 0.0, log);
        s2.run<double2>(*dev, t1.as<double2>(), t2.as<double2>(), log);
        s3.run<double2>(*dev, b->d(), t2.as<double2>(), out->d(), 1.0, 0.0, log);
    } else {
        DevBuf e32(dev->pool.get(), (size_t)env.lay.total * sizeof(float2));
        DevBuf k32(dev->pool.get(), (size_t)k->lay.total * sizeof(float2));
        DevBuf b32(dev->pool.get(), (size_t)b->lay.total * sizeof(float2));
        DevBuf o32(dev->pool.get(), (size_t)n3 * sizeof(float2));
        DevBuf t1(dev->pool.get(), n1 * sizeof(float2));
        DevBuf t2(dev->pool.get(), n2 * sizeof(float2));
        launch_f64_to_f32(dev->stream, env.d(), e32.as<float2>(), env.lay.total);
        launch_f64_to_f32(dev->stream, k->d(), k32.as<float2>(), k->lay.total);
        launch_f64_to_f32(dev->stream, b->d(), b32.as<float2>(), b->lay.total);
        s1.run<float2>(*dev, e32.as<float2>(), k32.as<float2>(), t1.as<float2>(), 1.0, 0.0, log);
        s2.run<float2>(*dev, t1.as<float2>(), t2.as<float2>(), log);
        s3.run<float2>(*dev, b32.as<float2>(), t2.as<float2>(), o32.as<float2>(), 1.0, 0.0, log);
        launch_f32_to_f64(dev->stream, o32.as<float2>(), out->d(), 1.0, n3);
    }
    Mark* done = log ? log->end() : nullptr;
    if (done) launch_mark(dev->stream, done);
    if (wait) dev->sync();
    return out;
}

}  // namespace kv
