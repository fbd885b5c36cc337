// Lanczos exponential of the effective Hamiltonian on the device, FP64 vector algebra.
// Follows local_krylov<Rank> (holstein/exponential.h:92-190) step by step:
//   v0 = x/|x| (:97-98); h = (dt/2) H_eff v_k (:113-125);
//   beta = <h|v_{k-1}> with the conjugate on h, as overlap(v_{k-1}, h) computes it, then
//   h -= beta v_{k-1} (:126-132); alpha = <h|v_k>, h -= alpha v_k (:134-137);
//   err *= |h|, stop when err < tol (:139-147); else v_{k+1} = h/|h| while
//   k < MaxIter-1 (:109, :156-159);  T = diag(alpha) + upper(beta), Hermitian
//   eigen-decomposition, c = V exp(-/+ i Lambda) V^H e_0 (:162-183);  x = sum c_i v_i
//   without renormalisation (:184-186).
// The H_eff contractions may run in complex FP32 (prec) from the second Krylov vector on;
// the first matvec and everything else in this file are FP64.
#pragma once

#include <chrono>
#include <complex>
#include <memory>
#include <vector>

#include "herm_eig.h"
#include "product.h"

namespace kv {

struct KrylovExit {
    bool converged = false;
    int iterations = 0;
    double error = 0;
    double loss_norm = 0;
};

struct LanczosStats {
    double heff_flop = 0;
    long matvecs = 0;
};

// x is replaced by exp(-/+ i dt/2 H_eff) x/|x| in H_eff's closed block layout.
inline KrylovExit local_krylov(const std::shared_ptr<Device>& dev, int nsite, const Tensor& L,
                               Tensor* W1, Tensor* W2, const Tensor& R,
                               std::unique_ptr<Tensor>& x, double dt, double tol, int max_iter,
                               bool reverse, Prec prec, MarkLog* log = nullptr,
                               LanczosStats* stats = nullptr, KernelStats* kstats = nullptr) {
    Heff H;
    H.build(dev, nsite, L, W1, W2, R, x->lay, prec);
    const Layout& xl = H.layout();
    const int64_t n = xl.total;
    const int nv_max = std::max(max_iter, 2);
    Device& D = *dev;
    std::unique_ptr<Tensor> spread;
    const Tensor* xin = x.get();
    if (!same_layout(x->lay, xl)) {
        spread = relayout(dev, *x, xl);
        xin = spread.get();
    }
    DevBuf V(D.pool.get(), (size_t)nv_max * (size_t)n * sizeof(double2));
    DevBuf hv(D.pool.get(), (size_t)n * sizeof(double2));
    DevBuf part(D.pool.get(), kLanczosPart * sizeof(double));
    double2* Vb = V.as<double2>();
    double2* h = hv.as<double2>();
    LanczosHost* rec = D.lanczos_host;
    const uint64_t tag = ++D.lanczos_calls << 8;
    launch_lanczos_begin(D.stream, xin->d(), Vb, n, part.as<double>(), D.lanczos_dev);

    // The recurrence and its stopping rule run on the device; the host queues iteration k + 1
    // before it reads the scalars of iteration k, and the launches of an iteration past the
    // last one return at once.
    auto queue = [&](int k) {
        // Mixed precision: the first matvec runs in FP64.  Its rounding error enters the
        // result at first order in dt/2 |H v|; the errors of later Krylov vectors are
        // damped by further powers of the Lanczos coefficients, so FP32 suffices there.
        double2* vk = Vb + (int64_t)k * n;
        H.apply(vk, h, dt * 0.5, log, k == 0, &D.lanczos_dev->stop[k]);
        launch_lanczos_step(D.stream, h, vk - n, vk, vk + n, n, part.as<double>(), D.lanczos_dev, k, tol, rec + k,
                            tag | (uint64_t)k, log ? log->end() : nullptr);
    };
    std::vector<std::complex<double>> alp, bet_up;
    double err = 1.0;
    KrylovExit ex;
    const int last = max_iter - 2;  // the last iteration the cap allows
    if (last >= 0 && err > tol) {
        queue(0);
        for (int k = 0;; ++k) {
            const size_t logged = log ? log->size() : 0;
            if (k < last) queue(k + 1);
            D.wait_record(rec[k], tag | (uint64_t)k);
            if (stats) {
                stats->heff_flop += H.flop();
                stats->matvecs += 1;
            }
            if (k > 0) bet_up.emplace_back(rec[k].beta_re, rec[k].beta_im);
            alp.emplace_back(rec[k].alpha_re, rec[k].alpha_im);
            err = rec[k].err;
            const bool stopped = !(err > tol);
            if (stopped && log) log->drop(logged);
            if (stopped || k == last) break;
        }
    }
    ex.converged = err < tol;
    ex.iterations = (int)alp.size();
    ex.error = err;
    std::vector<std::complex<double>> c = krylov_coefficients(alp, bet_up, reverse);
    auto out = Tensor::create(dev, xl, false);
    launch_lanczos_end(D.stream, out->d(), Vb, reinterpret_cast<const double2*>(c.data()), (int)c.size(), n,
                       part.as<double>(), rec + kLanczosMax, tag | 0xff);
    D.sync();
    if (log) log->resolve(kstats ? *kstats : D.stats);
    ex.loss_norm = 1.0 - std::sqrt(rec[kLanczosMax].nsq);
    x = std::move(out);
    return ex;
}

}  // namespace kv
