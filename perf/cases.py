"""The work that a user of this engine has it do, as cases that can be timed.

Kinds of case, each through the package's public entry points:

  krylov   one local time step of one tensor (local_krylov): exp(-+ i dt/2 H_eff) x on one
           site, two sites or a bond
  bond     one bond update as a sweep makes it: product, two-site local_krylov, svd_impl,
           env_sweep, the backward one-site local_krylov
  env      one environment update (env_sweep), also between two different states
  two      one two-site TDVP step of a chain from a given state (TDVP.two_site)
  one      one one-site TDVP step (TDVP.one_site)
  pp       one two-site step in the projected-purification layout, where every basis state
           is its own sector: many tiny blocks
  observe  C = <psi0|psi>, <psi|H|psi> and the exciton's population on every site
  grad     |C(T)|^2 of a one-site run and its gradient in all couplings (TdvpAutocorr)

Sizes are those of the repository's workloads: the 8-site chain with 8 levels at D <= 32, the
32-site chain with 16 levels at D = 256 (precision fp32, fp64), the batching set (8, 12 or 16
levels, caps 64..256), the two-mode sites (8 x 8 levels, split-BF16), the 24-site gradient.

Bond tensors are generated, not evolved, so that every input comes from the seed alone: the
centre bond carries a Schmidt spectrum that falls over five decades, the site tensors sit at
low phonon numbers, and the environments are what they are in a sweep (the identity on the
channel where no term has begun or all have ended, a Hermitian block Hamiltonian, the
exciton's hop between the charge sectors), so H_eff is Hermitian.

The factors of a truncated SVD are defined up to a unitary on the new bond.  Updated tensors
are therefore returned in the bond bases that the pass began with, as overlap_states
contracts them; nothing else is left out.  Where the H_eff contractions run in single
precision or split BF16 the result is taken as complex64.
"""
import math

import numpy as np
import torch

import __graft_entry__ as _entry

kv = _entry.load_package()
from kylin_v_amd import adjoint, model  # noqa: E402

LEFT, RIGHT, SITE = (1, -1, -1), (-1, 1, 1), (1, 1, -1)
CUTOFF, TOL, MAXITER = 1e-10, 1e-8, 15
W_DIMS = {-1: 1, 0: 2, 1: 1}  # MPO leg: open hop, (not begun, done), open hop


def listed():
    return [
        # a quick-start sized tensor: nothing but latency
        dict(name="krylov1_small", kind="krylov", nsite=1, L=4, modes=1, Dl=16, D=16, Dr=16, share=0.5,
             precision="fp64", reverse=False, dt=0.05),
        # two sites of a two-mode chain, whose bonds reach 34 in the 50-step run, split BF16
        dict(name="krylov2_two_mode", kind="krylov", nsite=2, L=8, modes=2, Dl=34, D=34, Dr=34, share=0.5,
             precision="bf16x3", reverse=False, dt=0.02),
        # one site of the two-mode chain at a wide bond, split BF16
        dict(name="krylov1_wide", kind="krylov", nsite=1, L=8, modes=2, Dl=192, D=192, Dr=192, share=0.5,
             precision="bf16x3", reverse=True, dt=0.02),
        # a bond of the 8-site chain at its cap
        dict(name="bond_small", kind="bond", L=8, modes=1, Dl=32, D=32, Dr=32, share=0.5, l2r=True,
             precision="fp64", dt=0.05),
        # a bond of one of the batched chains: odd sizes, sectors of different widths
        dict(name="bond_ragged", kind="bond", L=12, modes=1, Dl=97, D=101, Dr=103, share=0.57, l2r=False,
             precision="fp64", dt=0.05),
        # the middle bond of the 32-site chain, mixed precision and FP64, both directions
        dict(name="bond_mid_fp32", kind="bond", L=16, modes=1, Dl=256, D=256, Dr=256, share=0.5, l2r=True,
             precision="fp32", dt=0.02),
        dict(name="bond_mid_fp64", kind="bond", L=16, modes=1, Dl=256, D=256, Dr=256, share=0.5, l2r=False,
             precision="fp64", dt=0.02),
        # whole steps: the 8-site chain in both layouts, a one-site step of a longer chain
        dict(name="two_chain8", kind="two", N=8, L=8, modes=1, D=32, share=0.5, precision="fp64", dt=0.05),
        dict(name="pp_chain8", kind="pp", N=8, L=8, D=32, precision="fp64", dt=0.05),
        dict(name="one_chain12", kind="one", N=12, L=12, modes=1, D=64, share=0.5, precision="fp64", dt=0.05),
        # what is measured after a step of a longer chain
        dict(name="observe_chain16", kind="observe", N=16, L=16, modes=1, D=128, share=0.5),
        # the gradient, forward and backward
        dict(name="grad_chain6", kind="grad", N=6, L=6, D=16, steps=1, dt=0.05),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["krylov", "krylov", "bond", "bond", "bond", "env", "two", "one", "pp", "observe", "grad"])
    share, dt = round(rng.uniform(0.35, 0.65), 3), round(rng.uniform(0.01, 0.06), 4)
    precision = rng.choice(["fp64", "fp64", "fp32", "bf16x3"])
    if kind in ("krylov", "bond", "env"):
        modes = rng.choice([1, 1, 1, 2])
        L = rng.choice([4, 6, 8]) if modes == 2 else rng.choice([4, 7, 8, 11, 12, 16])
        P = L ** modes
        # the two-site tensor of the largest listed case bounds what is drawn
        hi = 256 if kind == "env" else min(256, int(256 * 16 / P))
        D = _log_int(rng, 12, hi)
        c = dict(kind=kind, L=L, modes=modes, Dl=min(hi, _log_int(rng, 0.8 * D, 1.25 * D)), D=D,
                 Dr=min(hi, _log_int(rng, 0.8 * D, 1.25 * D)), share=share)
        if kind == "krylov":
            nsite = rng.choice([0, 1, 1, 2])
            if nsite == 2 and (D * P) > 1500:
                c["D"] = c["Dl"] = c["Dr"] = max(4, 1500 // P + rng.randint(-2, 2))
            return dict(c, nsite=nsite, precision=precision, reverse=rng.random() < 0.3, dt=dt)
        if kind == "env":
            return dict(c, l2r=rng.random() < 0.5, bra=rng.random() < 0.3)
        return dict(c, l2r=rng.random() < 0.5, precision=precision, dt=dt)
    L = rng.choice([4, 6, 8, 10, 12])
    if kind == "pp":
        return dict(kind=kind, N=rng.randint(3, 8), L=rng.choice([4, 5, 6, 8]), D=rng.randint(8, 32),
                    precision="fp64", dt=dt)
    if kind == "grad":
        return dict(kind=kind, N=rng.randint(3, 6), L=rng.choice([3, 4, 6]), D=rng.randint(6, 16), steps=1, dt=dt)
    N, D = rng.randint(4, 12), _log_int(rng, 12, 64)
    if kind == "observe":
        return dict(kind=kind, N=rng.randint(4, 16), L=L, modes=1, D=_log_int(rng, 12, 128), share=share)
    if kind == "two":
        N, D = min(N, 8), min(D, 32)
    return dict(kind=kind, N=N, L=L, modes=1, D=D, share=share, precision="fp64", dt=dt)


# ---- inputs, as plain arrays ------------------------------------------------------------


def _split(D, share):
    d0 = min(D - 1, max(1, int(round(D * share)))) if D > 1 else 1
    return {0: d0, 1: D - d0} if D > d0 else {0: d0}


def _normal(rng, *shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


def _hermitian(rng, n):
    g = _normal(rng, n, max(1, n // 2))
    h = g @ g.conj().T
    return h * (2.0 / max(np.trace(h).real / n, 1e-300))


def _phonons(L, modes):
    """Number operator's diagonal and the sum of displacements of the site's modes, with the
    modes' frequencies (0.5, 1.5 for two of them)."""
    b = np.diag(np.sqrt(np.arange(1.0, L)), 1)
    omega = [0.5, 1.5][:modes]
    nb, x = np.zeros(L ** modes), np.zeros((L ** modes, L ** modes))
    count = np.zeros(L ** modes)
    for m in range(modes):
        l, r = np.eye(L ** m), np.eye(L ** (modes - 1 - m))
        n = np.diag(np.kron(np.kron(l, b.T @ b), r))
        nb, count = nb + omega[m] * n, count + n
        x = x + np.kron(np.kron(l, b + b.T), r)
    return nb, x, count


def _site_mpo(L, modes, g, J=1.0, left=True, right=True):
    """One site's MPO blocks (s', wL, s, wR) of the Holstein chain; charge of s: the exciton.
    left / right False: the chain ends on that side."""
    nb, x, _ = _phonons(L, modes)
    P = L ** modes
    eye = np.eye(P)
    lc = {(0, 0): ("start", "done")} if left else {(0, 0): ("start",)}
    rc = {(0, 0): ("start", "done")} if right else {(0, 0): ("done",)}
    lc, rc = dict(lc), dict(rc)
    if left:
        lc[(-1, 0)], lc[(1, 0)] = ("down",), ("up",)
    if right:
        rc[(-1, 0)], rc[(1, 0)] = ("down",), ("up",)
    local = {0: np.diag(nb), 1: np.diag(nb) + g * x}
    terms = {("start", "start"): {(0, 0): eye, (1, 1): eye}, ("done", "done"): {(0, 0): eye, (1, 1): eye},
             ("start", "done"): {(0, 0): local[0], (1, 1): local[1]},
             ("start", "up"): {(1, 0): J * eye}, ("up", "done"): {(0, 1): eye},
             ("start", "down"): {(0, 1): J * eye}, ("down", "done"): {(1, 0): eye}}
    out = {}
    for (ql, _), ln in lc.items():
        for (qr, _), rn in rc.items():
            for i, a in enumerate(ln):
                for j, b in enumerate(rn):
                    for (sp, s), m in terms.get((a, b), {}).items():
                        key = (sp, ql, s, qr)
                        out.setdefault(key, np.zeros((P, len(ln), P, len(rn)), complex))[:, i, :, j] += m
    return out


def _number_mpo(L, modes, here):
    """One site of the exciton number's product operator: n where `here`, else the identity."""
    eye = np.eye(L ** modes).reshape(L ** modes, 1, L ** modes, 1).astype(complex)
    return {(1, 0, 1, 0): eye} if here else {(0, 0, 0, 0): eye, (1, 0, 1, 0): eye}


def _isometry(rng, left, right, P, weight, to_right):
    """Site blocks (a, s, b) with orthonormal columns over (a, s) (to_right) or orthonormal rows
    over (s, b), small at high phonon numbers."""
    out = {}
    for q in sorted(right if to_right else left):
        keys = [(q - s, s, q) if to_right else (q, s, q + s) for s in (0, 1)]
        keys = [k for k in keys if k[0] in left and k[2] in right]
        n = right[q] if to_right else left[q]
        sizes = [(left[k[0]] if to_right else right[k[2]]) for k in keys]
        m = [(_normal(rng, d, P, n) * weight[None, :, None]).reshape(d * P, n) for d in sizes]
        u, _ = np.linalg.qr(np.concatenate(m))
        at = 0
        for k, d in zip(keys, sizes):
            blk = u[at:at + d * P].reshape(d, P, n)
            at += d * P
            out[k] = np.ascontiguousarray(blk if to_right else blk.transpose(2, 1, 0))
    return out


def _environment(rng, dims, side):
    """(a', w, a): the identity where no term is open, a Hermitian block Hamiltonian, and the hop
    between the sectors, as the left (side 0) or right (side 1) environment of a bond."""
    out = {}
    for q, n in dims.items():
        blk = np.zeros((n, 2, n), complex)
        blk[:, side, :] = np.eye(n)
        blk[:, 1 - side, :] = _hermitian(rng, n)
        out[(q, 0, q)] = blk
    if len(dims) == 2:
        k = _normal(rng, dims[1], dims[0]) / (2.0 * (math.sqrt(dims[0]) + math.sqrt(dims[1])))
        out[(1, 1, 0)] = k[:, None, :].copy()
        out[(0, -1, 1)] = k.conj().T[:, None, :].copy()
    return out


def _fit(dims, left, right, P):
    """The centre bond's sectors, no wider than the sites beside it can fill."""
    fit = {}
    for q, n in dims.items():
        rows = P * sum(left.get(q - s, 0) for s in (0, 1))
        cols = P * sum(right.get(q + s, 0) for s in (0, 1))
        if min(rows, cols) > 0:
            fit[q] = min(n, rows, cols)
    return fit


def _bond(case, seed):
    rng = np.random.default_rng([int(seed), 11])
    P = case["L"] ** case["modes"]
    dl, dr = _split(case["Dl"], case["share"]), _split(case["Dr"], case["share"])
    dc = _fit(_split(case["D"], case["share"]), dl, dr, P)
    weight = np.exp(-0.5 * _phonons(case["L"], case["modes"])[2])
    g = rng.uniform(0.7, 1.2, 2)
    spectrum = {q: 10.0 ** (-5.0 * (np.arange(n) + rng.random(n)) / n) * (1.0 if q == 0 else 0.6)
                for q, n in dc.items()}
    norm = math.sqrt(sum(float(v @ v) for v in spectrum.values()))
    return dict(legs=dict(l=dl, c=dc, r=dr), P=P,
                L=_environment(rng, dl, 0), R=_environment(rng, dr, 1),
                A=_isometry(rng, dl, dc, P, weight, True), B=_isometry(rng, dc, dr, P, weight, False),
                lam={q: v / norm for q, v in spectrum.items()},
                W1=_site_mpo(case["L"], case["modes"], g[0]), W2=_site_mpo(case["L"], case["modes"], g[1]))


def _weighted(site, lam, on_right):
    if on_right:
        return {k: b * lam[k[2]][None, None, :] for k, b in site.items()}
    return {k: b * lam[k[0]][:, None, None] for k, b in site.items()}


def _chain(case, seed):
    """Right-canonical chain with one exciton, its centre on site 0; couplings of its MPO."""
    rng = np.random.default_rng([int(seed), 12])
    N, P = case["N"], case["L"] ** case["modes"]
    weight = np.exp(-0.7 * _phonons(case["L"], case["modes"])[2])
    bonds = [{0: 1}]
    for i in range(1, N):
        cap = _split(case["D"], case["share"])
        room = {0: min(P ** min(i, 8), (N - i) * P ** min(N - i, 8)), 1: min(i * P ** min(i, 8), P ** min(N - i, 8))}
        bonds.append({q: min(cap[q], room[q]) for q in cap})
    bonds.append({1: 1})
    for i in reversed(range(1, N)):
        for q in bonds[i]:
            bonds[i][q] = min(bonds[i][q], P * sum(bonds[i + 1].get(q + s, 0) for s in (0, 1)))
    sites = [_isometry(rng, bonds[i], bonds[i + 1], P, weight, False) for i in range(N)]
    # a physical bond spectrum falls off: damp the later states of every bond, then restore the
    # canonical form site by site from the right
    for i in reversed(range(1, N)):
        rows = {}
        for (a, s, b), blk in sites[i].items():
            if i + 1 < N:
                blk = blk * (10.0 ** (-3.0 * np.arange(blk.shape[2]) / blk.shape[2]))[None, None, :]
            rows.setdefault(a, []).append((s, b, blk))
        for a, parts in rows.items():
            m = np.concatenate([blk.reshape(blk.shape[0], -1) for _, _, blk in parts], axis=1)
            u, _ = np.linalg.qr(m.conj().T)
            at = 0
            for s, b, blk in parts:
                n = blk[0].size
                sites[i][(a, s, b)] = u[at:at + n].conj().T.reshape(blk.shape).copy()
                at += n
    first = {k: b * (10.0 ** (-3.0 * np.arange(b.shape[2]) / b.shape[2]))[None, None, :] for k, b in sites[0].items()}
    n = math.sqrt(sum(float(np.vdot(b, b).real) for b in first.values()))
    sites[0] = {k: b / n for k, b in first.items()}
    g = rng.uniform(0.8, 1.2, N)
    mpo = [_site_mpo(case["L"], case["modes"], g[i], left=i > 0, right=i < N - 1) for i in range(N)]
    return sites, mpo


# ---- what a program has in hand -----------------------------------------------------------


def _up(dirs, blocks):
    return kv.Tensor.from_blocks(dirs, blocks)


def _mpo(blocks):
    return _up((1, 1, -1, -1), blocks)


def prepare(case, seed):
    kind = case["kind"]
    st = dict(case=case)
    if kind in ("krylov", "bond", "env"):
        b = _bond(case, seed)
        st.update(L=_up(LEFT, b["L"]), R=_up(RIGHT, b["R"]), W1=_mpo(b["W1"]), W2=_mpo(b["W2"]))
        A, B = _up(SITE, b["A"]), _up(SITE, b["B"])
        if kind == "env":
            st["ket"] = _up(SITE, _weighted(b["A"], b["lam"], True) if not case["l2r"] else b["A"])
            if not case["l2r"]:  # the updated site ends at the centre bond
                st["R"] = _up(RIGHT, _centre_env(case, seed, 1))
            st["bra"] = None
            if case["bra"]:
                o = _bond(case, seed + 1000003)
                st["bra"] = _up(SITE, o["A"])
        elif kind == "krylov":
            n = case["nsite"]
            centre = _up(SITE, _weighted(b["A"], b["lam"], True))
            if n == 0:
                st["x"] = _up((1, -1), {(q, q): np.diag(v).astype(complex) for q, v in b["lam"].items()})
                st["L"], st["R"] = _up(LEFT, _centre_env(case, seed, 0)), _up(RIGHT, _centre_env(case, seed, 1))
            elif n == 1:
                st["x"] = centre
                st["R"] = _up(RIGHT, _centre_env(case, seed, 1))
            else:
                st["x"] = kv.product(centre, B, 1)
        else:
            l2r = case["l2r"]
            st["A"] = _up(SITE, _weighted(b["A"], b["lam"], True)) if l2r else A
            st["B"] = B if l2r else _up(SITE, _weighted(b["B"], b["lam"], False))
            st["basis"] = A if l2r else B
    elif kind in ("two", "one", "observe"):
        sites, mpo = _chain(case, seed)
        st["mps"], st["mpo"] = [_up(SITE, s) for s in sites], [_mpo(w) for w in mpo]
        if kind == "observe":
            other, _ = _chain(case, seed + 1000003)
            st["psi0"] = [_up(SITE, s) for s in other]
            off, on = (_mpo(_number_mpo(case["L"], case["modes"], here)) for here in (False, True))
            st["numbers"] = [[on if j == i else off for j in range(case["N"])] for i in range(case["N"])]
    elif kind == "pp":
        rng = np.random.default_rng([int(seed), 13])
        ch = model.HolsteinChain(case["N"], [1.0], rng.uniform(0.8, 1.2, case["N"]), [case["L"]], 1.0, "pp")
        eng = kv.TDVP(ch.psi0, ch.mpo, cutoff=CUTOFF, maxdim=case["D"], dt=case["dt"])
        for _ in range(2):  # the global Krylov steps open the sectors that the sweeps need
            eng.global_krylov()
        for _ in range(2):
            eng.two_site()
        st["mps"], st["mpo"], st["chain"] = eng.mps, ch.mpo, ch
    else:
        rng = np.random.default_rng([int(seed), 14])
        N = case["N"]
        sites, _, init, _ = model.chain(N, [1.0], np.ones((N, 1)), [case["L"]], 1.0, "merged")
        psi0 = model.expanded_state_blocks(sites, init, D=case["D"], seed=int(seed), eps=0.2)
        st["engine"] = adjoint.OneSiteAdjoint(N, case["L"], case["dt"], case["steps"], psi0,
                                              adjoint.DeviceOps(kv.default_context()))
        st["theta"] = torch.tensor([*rng.uniform(0.8, 1.2, N), 1.0, 1.0], dtype=torch.float64, requires_grad=True)
    return st


def _centre_env(case, seed, side):
    rng = np.random.default_rng([int(seed), 15 + side])
    return _environment(rng, _bond_legs(case)["c"], side)


def _bond_legs(case):
    P = case["L"] ** case["modes"]
    dl, dr = _split(case["Dl"], case["share"]), _split(case["Dr"], case["share"])
    return dict(l=dl, c=_fit(_split(case["D"], case["share"]), dl, dr, P), r=dr)


# ---- one pass -----------------------------------------------------------------------------


def _taken(t, case):
    a = t.download()
    return a if case.get("precision", "fp64") == "fp64" else a.astype(np.complex64)


def _copy(t):
    return kv.transpose(t, range(t.rank))


def _framed(old, new, Q):
    """The tensors of the state `new` in the bond bases of `old`."""
    n = len(old)
    left = [_up((1, -1), {(0, 0): np.ones((1, 1), complex)})]
    right = [_up((1, -1), {(Q, Q): np.ones((1, 1), complex)})]
    for i in range(n - 1):
        left.append(kv.product(old[i], kv.product(left[-1], new[i], 1), 2, "C", "N"))
    for i in range(n - 1, 0, -1):
        right.append(kv.product(kv.product(new[i], right[-1], 1), old[i], 2, "N", "C"))
    right.reverse()
    return [kv.product(kv.product(left[i], new[i], 1), right[i], 1) for i in range(n)]


def run(st):
    case = st["case"]
    kind = case["kind"]
    if kind == "krylov":
        W1, W2 = (st["W1"] if case["nsite"] else None), (st["W2"] if case["nsite"] == 2 else None)
        x, _ = kv.local_krylov(st["L"], _copy(st["x"]), W1, W2, st["R"], case["dt"], TOL, MAXITER,
                               reverse=case["reverse"], nsite=case["nsite"], precision=case["precision"])
        return _taken(x, case)
    if kind == "bond":
        l2r, dt, prec = case["l2r"], case["dt"], case["precision"]
        x = kv.product(st["A"], st["B"], 1)
        x, _ = kv.local_krylov(st["L"], x, st["W1"], st["W2"], st["R"], dt, TOL, MAXITER, precision=prec)
        left, right = kv.svd_impl(x, 2, CUTOFF, case["D"], l2r)
        if l2r:
            env = kv.env_sweep(st["L"], left, st["W1"], True)
            y, _ = kv.local_krylov(env, right, st["W2"], None, st["R"], dt, TOL, MAXITER, reverse=True, precision=prec)
            y = kv.product(kv.product(st["basis"], left, 2, "C", "N"), y, 1)
        else:
            env = kv.env_sweep(st["R"], right, st["W2"], False)
            y, _ = kv.local_krylov(st["L"], left, st["W1"], None, env, dt, TOL, MAXITER, reverse=True, precision=prec)
            y = kv.product(y, kv.product(right, st["basis"], 2, "N", "C"), 1)
        return _taken(y, case)
    if kind == "env":
        ket, bra = st["ket"], st["bra"]
        if case["l2r"]:
            return kv.env_sweep(st["L"], ket, st["W1"], True, bra=bra).download()
        return kv.env_sweep(st["R"], ket, st["W1"], False, bra=bra).download()
    if kind in ("two", "one", "pp"):
        eng = kv.TDVP(st["mps"], st["mpo"], cutoff=CUTOFF, maxdim=case["D"], dt=case["dt"],
                      precision=case["precision"])
        if kind == "one":
            eng.one_site()
        else:
            eng.two_site()
        new = eng.mps
        out = [kv.overlap_states(st["mps"], new)]
        out = [out[0].real, out[0].imag]
        if kind == "pp":
            pops = [kv.join(st["chain"].density(i), new, new).real for i in range(case["N"])]
            return out + [np.array(pops), kv.join(st["mpo"], new, new).real]
        return out + [_taken(t, case) for t in _framed(st["mps"], new, 1)]
    if kind == "observe":
        c = kv.overlap_states(st["psi0"], st["mps"])
        e = kv.join(st["mpo"], st["mps"], st["mps"])
        n = [kv.join(w, st["mps"], st["mps"]).real for w in st["numbers"]]
        return [np.array([c.real, c.imag]), np.array([e.real]), np.array(n)]
    theta = st["theta"]
    theta.grad = None
    loss = adjoint.TdvpAutocorr.apply(theta, st["engine"])
    loss.backward()
    return [loss.detach().clone(), theta.grad.clone()]


# ---- what a pass cannot do without ----------------------------------------------------------


def _heff_flops(legs_l, legs_r, P, nsite):
    """8 m n k of L x and (L W x) R^T over the charge blocks."""
    total = 0.0
    for q, n in legs_l.items():
        for moved in range(nsite + 1):
            b = q + moved
            if b not in legs_r:
                continue
            site = P ** nsite * (math.comb(nsite, moved))
            total += 8.0 * site * n * legs_r[b] * sum(W_DIMS[w] * legs_l.get(q + w, 0) for w in W_DIMS)
            total += 8.0 * site * n * legs_r[b] * sum(W_DIMS[w] * legs_r.get(b - w, 0) for w in W_DIMS)
    return total


def _elems(legs_l, legs_r, P, nsite):
    return float(sum(n * legs_r.get(q + m, 0) * math.comb(nsite, m) * P ** nsite
                     for q, n in legs_l.items() for m in range(nsite + 1)))


def _env_elems(legs):
    return float(sum(W_DIMS[w] * n * legs.get(q + w, 0) for q, n in legs.items() for w in W_DIMS))


def _bond_flops(l, c, r, P, lanczos=6):
    theta, site = _elems(l, r, P, 2), _elems(l, c, P, 1)
    kept = sum(c.values()) / max(len(c), 1)
    return (8.0 * theta * kept + lanczos * (_heff_flops(l, r, P, 2) + _heff_flops(c, r, P, 1))
            + 4 * 8.0 * theta * kept + 2 * 8.0 * site * kept)


def work(case):
    kind = case["kind"]
    if kind in ("krylov", "bond", "env"):
        P = case["L"] ** case["modes"]
        d = _bond_legs(case)
        l, c, r = d["l"], d["c"], d["r"]
        site_l, site_r = _elems(l, c, P, 1), _elems(c, r, P, 1)
        if kind == "env":
            return dict(bytes=16.0 * (_env_elems(l) + _env_elems(c) + (2 if case["bra"] else 1) * site_l),
                        flops=_heff_flops(l, c, P, 1))
        if kind == "krylov":
            a, b = {0: (c, c), 1: (l, c), 2: (l, r)}[case["nsite"]]
            x = _elems(a, b, P, case["nsite"])
            return dict(bytes=16.0 * (_env_elems(a) + _env_elems(b) + 2 * x),
                        flops=6 * _heff_flops(a, b, P, case["nsite"]))
        return dict(bytes=16.0 * (_env_elems(l) + _env_elems(r) + 2 * (site_l + site_r)),
                    flops=_bond_flops(l, c, r, P))
    N, L = case["N"], case["L"]
    P = L ** case.get("modes", 1)
    d = _split(case["D"], case.get("share", 0.5))
    site = _elems(d, d, P, 1)
    if kind == "observe":
        return dict(bytes=16.0 * N * 2 * site, flops=(N + 1) * N * _heff_flops(d, d, P, 1) / 4)
    if kind == "pp":  # 3 N sites of one-dimensional basis states, bonds of D over the charges
        return dict(bytes=16.0 * 3 * N * 2 * case["D"] * L, flops=2.0 * 3 * N * 12 * 8 * 4 * case["D"] ** 2 * L)
    steps = 2.0 * (N - 1)
    if kind == "two":
        return dict(bytes=16.0 * N * 2 * site, flops=steps * _bond_flops(d, d, d, P))
    one = steps * 6 * (_heff_flops(d, d, P, 1) + _heff_flops(d, d, P, 0))
    if kind == "one":
        return dict(bytes=16.0 * N * 2 * site, flops=one)
    return dict(bytes=16.0 * N * 2 * site * case["steps"], flops=5 * one * case["steps"])


# ---- the same in 64 bits with plain torch -----------------------------------------------------


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _at(leg, q):
    """Where sector q sits in a dense leg with sectors in ascending charge."""
    lo = sum(n for p, n in leg.items() if p < q)
    return slice(lo, lo + leg[q])


def _dense(blocks, legs):
    legs = [dict(sorted(leg.items())) for leg in legs]
    t = torch.zeros([sum(leg.values()) for leg in legs], dtype=torch.complex128)
    for key, blk in blocks.items():
        t[tuple(_at(leg, q) for leg, q in zip(legs, key))] = torch.from_numpy(np.ascontiguousarray(blk))
    return t.to(_device())


def _flat(t, legs, dirs):
    """The blocks of a dense tensor that charge allows, in ascending charges, as one array."""
    parts = []

    def walk(i, key):
        if i == len(legs):
            if sum(d * q for d, q in zip(dirs, key)) == 0:
                parts.append(t[tuple(_at(leg, q) for leg, q in zip(legs, key))].reshape(-1))
            return
        for q in sorted(legs[i]):
            walk(i + 1, key + (q,))

    walk(0, ())
    return torch.cat(parts).cpu().numpy()


def _heff(L, W, R, x):
    """L W x R on a dense tensor with as many site legs as W has tensors."""
    n = len(W)
    t = torch.tensordot(L, x, ([2], [0]))  # a' w s.. b
    if n == 0:
        return torch.tensordot(t, R, ([2, 1], [2, 1]))
    t = torch.tensordot(t, W[0], ([1, 2], [1, 2]))  # a' (s2) b s1' w
    if n == 2:
        t = torch.tensordot(t, W[1], ([4, 1], [1, 2]))  # a' b s1' s2' w
    return torch.tensordot(t, R, ([1, t.dim() - 1], [2, 1]))


def _expm(L, W, R, x, dt, reverse):
    v = [x / torch.linalg.vector_norm(x)]
    alpha, beta, err = [], [], 1.0
    for k in range(MAXITER - 1):
        h = _heff(L, W, R, v[k]) * (0.5 * dt)
        if k:
            beta.append(complex(torch.vdot(h.reshape(-1), v[k - 1].reshape(-1))))
            h = h - beta[-1] * v[k - 1]
        alpha.append(complex(torch.vdot(h.reshape(-1), v[k].reshape(-1))))
        h = h - alpha[-1] * v[k]
        nrm = float(torch.linalg.vector_norm(h))
        err *= nrm
        if err < TOL:
            break
        if k + 1 < MAXITER - 1:
            v.append(h / nrm)
    m = len(alpha)
    T = np.diag(np.array(alpha)) + np.diag(np.array(beta[:m - 1]), 1)
    T = np.triu(T) + np.triu(T, 1).conj().T
    T = T - 1j * np.diag(np.diag(T).imag)
    w, Z = np.linalg.eigh(T)
    c = Z @ (np.exp((1j if reverse else -1j) * w) * Z[0].conj())
    return sum(complex(ci) * vi for ci, vi in zip(c, v))


def _env_left(E, bra, W, ket):
    t = torch.tensordot(E, ket, ([2], [0]))  # a' w s b
    t = torch.tensordot(t, W, ([1, 2], [1, 2]))  # a' b s' w2
    return torch.tensordot(bra.conj(), t, ([0, 1], [0, 2])).permute(0, 2, 1).contiguous()


def _env_right(E, bra, W, ket):
    t = torch.tensordot(ket, E, ([2], [2]))  # a s b' wR
    t = torch.tensordot(t, W, ([1, 3], [2, 3]))  # a b' s' wL
    return torch.tensordot(bra.conj(), t, ([1, 2], [2, 1])).permute(0, 2, 1).contiguous()


def _charges(leg):
    return np.concatenate([np.full(n, q) for q, n in sorted(leg.items())])


def _truncated(x, rows, cols, r1, maxdim, l2r):
    """(left, right, bond leg) of the truncated SVD of a dense tensor, rows: the legs left of the
    cut (charges add up to the bond's), cols: (leg, sign) right of it."""
    m = x.reshape(int(np.prod(x.shape[:r1])), -1)
    rq = np.add.outer(*map(_charges, rows)).ravel() if r1 == 2 else _charges(rows[0])
    signed = [s * _charges(leg) for leg, s in cols]
    cq = np.add.outer(*signed).ravel() if len(cols) == 2 else signed[0]
    parts = []
    for q in sorted(set(rq) & set(cq)):
        i, j = np.nonzero(rq == q)[0], np.nonzero(cq == q)[0]
        blk = m[torch.from_numpy(i).to(m.device)][:, torch.from_numpy(j).to(m.device)]
        if min(blk.shape) > 1000:
            wide = blk.shape[1] >= blk.shape[0]
            w, z = torch.linalg.eigh(blk @ blk.mH if wide else blk.mH @ blk)
            w, z = w.flip(0)[:maxdim], z.flip(1)[:, :maxdim]
            s = torch.sqrt(w.clamp_min(0))
            u, v = (z, (z.mH @ blk) / s[:, None]) if wide else ((blk @ z) / s[None, :], z.mH)
            s = s.cpu().numpy()
        else:
            u, s, v = np.linalg.svd(blk.cpu().numpy(), full_matrices=False)
            u, v = torch.from_numpy(u).to(m.device), torch.from_numpy(v).to(m.device)
        parts.append((int(q), i, j, u, s, v))
    every = sorted(((float(s), k, n) for k, p in enumerate(parts) for n, s in enumerate(p[4])), key=lambda e: -e[0])
    kept = [e for n, e in enumerate(every) if n == 0 or (n < maxdim and e[0] > CUTOFF)]
    leg = {p[0]: sum(1 for e in kept if e[1] == k) for k, p in enumerate(parts)}
    leg = {q: n for q, n in leg.items() if n}
    D = sum(leg.values())
    left = torch.zeros((m.shape[0], D), dtype=m.dtype, device=m.device)
    right = torch.zeros((D, m.shape[1]), dtype=m.dtype, device=m.device)
    for q, i, j, u, s, v in parts:
        if q not in leg:
            continue
        k, at = leg[q], _at(leg, q)
        sv = torch.from_numpy(np.asarray(s[:k], complex)).to(m.device)
        left[torch.from_numpy(i).to(m.device), at] = u[:, :k] * (1 if l2r else sv[None, :])
        right[at, torch.from_numpy(j).to(m.device)] = (sv[:, None] if l2r else 1) * v[:k]
    return left.reshape(*x.shape[:r1], D), right.reshape(D, *x.shape[r1:]), leg


def _mps_dense(sites):
    legs = [dict() for _ in range(len(sites) + 1)]
    for i, s in enumerate(sites):
        for (a, _, b), blk in s.items():
            legs[i][a], legs[i + 1][b] = blk.shape[0], blk.shape[2]
    return legs


def _mpo_dense(blocks, P):
    left = {k[1]: b.shape[1] for k, b in blocks.items()}
    right = {k[3]: b.shape[3] for k, b in blocks.items()}
    site = {0: P, 1: P}
    return _dense(blocks, [site, left, site, right])


def _one():
    return torch.ones((1, 1, 1), dtype=torch.complex128, device=_device())


def _exact_step(case, sites, mpo):
    P, D, dt, n = case["L"] ** case["modes"], case["D"], case["dt"], case["N"]
    site = {0: P, 1: P}
    legs = _mps_dense(sites)
    old_legs = list(legs)
    old = [_dense(s, [legs[i], site, legs[i + 1]]) for i, s in enumerate(sites)]
    W = [_mpo_dense(w, P) for w in mpo]
    M, R = list(old), {n: _one()}
    for i in range(n - 1, 0, -1):
        R[i] = _env_right(R[i + 1], M[i], W[i], M[i])
    Le = {0: _one()}
    if case["kind"] == "two":
        for l2r in (True, False):
            for i in (range(n - 1) if l2r else range(n - 2, -1, -1)):
                x = _expm(Le[i], [W[i], W[i + 1]], R[i + 2], torch.tensordot(M[i], M[i + 1], 1), dt, False)
                a, b, legs[i + 1] = _truncated(x, [legs[i], site], [(site, -1), (legs[i + 2], 1)], 2, D, l2r)
                if l2r:
                    Le[i + 1] = _env_left(Le[i], a, W[i], a)
                    if i < n - 2:
                        b = _expm(Le[i + 1], [W[i + 1]], R[i + 2], b, dt, True)
                else:
                    R[i + 1] = _env_right(R[i + 2], b, W[i + 1], b)
                    if i > 0:
                        a = _expm(Le[i], [W[i]], R[i + 1], a, dt, True)
                M[i], M[i + 1] = a, b
    else:
        for l2r in (True, False):
            for i in (range(n) if l2r else range(n - 1, -1, -1)):
                x = _expm(Le[i], [W[i]], R[i + 1], M[i], dt, False)
                if l2r and i < n - 1:
                    M[i], c, legs[i + 1] = _truncated(x, [legs[i], site], [(legs[i + 1], 1)], 2, D, True)
                    Le[i + 1] = _env_left(Le[i], M[i], W[i], M[i])
                    M[i + 1] = torch.tensordot(_expm(Le[i + 1], [], R[i + 1], c, dt, True), M[i + 1], 1)
                elif not l2r and i > 0:
                    c, M[i], legs[i] = _truncated(x, [legs[i]], [(site, -1), (legs[i + 1], 1)], 1, D, False)
                    R[i] = _env_right(R[i + 1], M[i], W[i], M[i])
                    M[i - 1] = torch.tensordot(M[i - 1], _expm(Le[i], [], R[i], c, dt, True), 1)
                else:
                    M[i] = x
    one = torch.ones((1, 1), dtype=torch.complex128, device=_device())
    left, right = [one], [one]
    for i in range(n - 1):
        left.append(torch.tensordot(old[i].conj(), torch.tensordot(left[-1], M[i], 1), ([0, 1], [0, 1])))
    for i in range(n - 1, 0, -1):
        right.append(torch.tensordot(torch.tensordot(M[i], right[-1], 1), old[i].conj(), ([1, 2], [1, 2])))
    right.reverse()
    framed = [torch.tensordot(torch.tensordot(left[i], M[i], 1), right[i], 1) for i in range(n)]
    c = complex(torch.vdot(old[n - 1].reshape(-1), torch.tensordot(left[n - 1], M[n - 1], 1).reshape(-1)))
    return [c.real, c.imag] + [_flat(t, [old_legs[i], site, old_legs[i + 1]], SITE) for i, t in enumerate(framed)]


def exact(case, seed):
    kind = case["kind"]
    if kind in ("pp", "grad"):
        return None
    P = case["L"] ** case["modes"]
    site = {0: P, 1: P}
    if kind in ("krylov", "bond", "env"):
        b = _bond(case, seed)
        l, c, r = b["legs"]["l"], b["legs"]["c"], b["legs"]["r"]
        W1, W2 = _mpo_dense(b["W1"], P), _mpo_dense(b["W2"], P)
        Le, R = _dense(b["L"], [l, W_DIMS, l]), _dense(b["R"], [r, W_DIMS, r])
        A, B = _dense(b["A"], [l, site, c]), _dense(b["B"], [c, site, r])
        lam = torch.cat([torch.from_numpy(b["lam"][q]) for q in sorted(b["lam"])]).to(_device()).to(torch.complex128)
        if kind == "env":
            other = _dense(_bond(case, seed + 1000003)["A"], [l, site, c]) if case["bra"] else None
            if case["l2r"]:
                return _flat(_env_left(Le, A if other is None else other, W1, A), [c, W_DIMS, c], LEFT)
            ket = A * lam[None, None, :]
            Rc = _dense(_centre_env(case, seed, 1), [c, W_DIMS, c])
            return _flat(_env_right(Rc, ket if other is None else other, W1, ket), [l, W_DIMS, l], RIGHT)
        if kind == "krylov":
            n = case["nsite"]
            if n == 0:
                Le = _dense(_centre_env(case, seed, 0), [c, W_DIMS, c])
            if n < 2:
                R = _dense(_centre_env(case, seed, 1), [c, W_DIMS, c])
            x = {0: lambda: torch.diag(lam), 1: lambda: A * lam[None, None, :],
                 2: lambda: torch.tensordot(A * lam[None, None, :], B, 1)}[n]()
            y = _expm(Le, [W1, W2][:n], R, x, case["dt"], case["reverse"])
            return _flat(y, *{0: ([c, c], (1, -1)), 1: ([l, site, c], SITE),
                              2: ([l, site, site, r], (1, 1, 1, -1))}[n])
        l2r, dt = case["l2r"], case["dt"]
        x = _expm(Le, [W1, W2], R, torch.tensordot(A * lam[None, None, :], B, 1), dt, False)
        left, right, _ = _truncated(x, [l, site], [(site, -1), (r, 1)], 2, case["D"], l2r)
        del x
        if l2r:
            y = _expm(_env_left(Le, left, W1, left), [W2], R, right, dt, True)
            y = torch.tensordot(torch.tensordot(A.conj(), left, ([0, 1], [0, 1])), y, 1)
            return _flat(y, [c, site, r], SITE)
        y = _expm(Le, [W1], _env_right(R, right, W2, right), left, dt, True)
        y = torch.tensordot(y, torch.tensordot(right, B.conj(), ([1, 2], [1, 2])), 1)
        return _flat(y, [l, site, c], SITE)
    sites, mpo = _chain(case, seed)
    if kind in ("two", "one"):
        return _exact_step(case, sites, mpo)
    legs = _mps_dense(sites)
    ket = [_dense(s, [legs[i], site, legs[i + 1]]) for i, s in enumerate(sites)]
    other, _ = _chain(case, seed + 1000003)
    bra = [_dense(s, [legs[i], site, legs[i + 1]]) for i, s in enumerate(other)]

    def value(ws, left):
        e = _one()
        for w, a, m in zip(ws, left, ket):
            e = _env_left(e, a, w, m)
        return complex(e.reshape(-1)[0])

    off, on = (_mpo_dense(_number_mpo(case["L"], case["modes"], here), P) for here in (False, True))
    c = value([off] * case["N"], bra)
    e = value([_mpo_dense(w, P) for w in mpo], ket)
    n = [value([on if j == i else off for j in range(case["N"])], ket).real for i in range(case["N"])]
    return [np.array([c.real, c.imag]), np.array([e.real]), np.array(n)]
