"""Each path of a dispatch against plain FP64 numpy at the sizes where the path changes."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import __graft_entry__ as GE  # noqa: E402

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -52


def cplx(rng, *shape):
    return rng.standard_normal(shape) + 1j * rng.standard_normal(shape)


# (m, n, K dims of the contracted leg's sectors): whole K, two chunks, the chunk limits on
# either side, odd K that no chunk divides, sectors far shorter than the others, many tiles
SPLIT = [(5, 7, [127]), (64, 64, [128]), (65, 3, [129]), (1, 1, [2048, 1]), (70, 130, [1000, 1047]),
         (33, 17, [3, 4099, 200]), (513, 520, [260])]


@pytest.mark.parametrize("m,n,ks", SPLIT)
@pytest.mark.parametrize("ops", ["NN", "NT", "NC", "CN"])
def test_product_with_a_deep_k(m, n, ks, ops):
    kv = GE.load_package()
    rng = np.random.default_rng([m, n, len(ks)])
    print(f"case product {ops} {m}x{n} K {ks}", flush=True)
    # contracted legs (carried, summed) with carried = summed: every sector of the summed leg
    # adds to the one output block
    A, B = [cplx(rng, m, k) for k in ks], [cplx(rng, k, n) for k in ks]
    if ops[0] == "N":
        ta = kv.Tensor.from_blocks((1, 1, -1), {(0, q, q): a[:, None, :] for q, a in enumerate(A)})
    else:
        ta = kv.Tensor.from_blocks((-1, 1, 1), {(q, q, 0): a.conj().T[None] for q, a in enumerate(A)})
    if ops[1] == "N":
        tb = kv.Tensor.from_blocks((-1, 1, 1), {(q, q, 0): b[None] for q, b in enumerate(B)})
    elif ops[1] == "T":
        tb = kv.Tensor.from_blocks((1, -1, 1), {(0, q, q): b.T[:, None, :] for q, b in enumerate(B)})
    else:
        tb = kv.Tensor.from_blocks((1, 1, -1), {(0, q, q): b.conj().T[:, None, :] for q, b in enumerate(B)})
    (got,) = kv.product(ta, tb, 2, *ops).to_blocks()[1].values()
    ref = sum(a @ b for a, b in zip(A, B))
    mag = sum(abs(a) @ abs(b) for a, b in zip(A, B))
    # two roundings per real product and sum, on either side of the comparison
    assert np.all(abs(got.reshape(m, n) - ref) <= 4 * (sum(ks) + 8) * EPS * mag)


# one-workgroup iterations of one, two and three chunks per wave and their limits, the first
# sizes of the multi-launch form, a vector shorter than a chunk; D, P, levels of the bond
LANCZOS = [(1, 1, 1), (3, 2, 5), (32, 4, 32), (33, 4, 32), (32, 8, 32), (33, 8, 32), (32, 12, 32), (33, 12, 32),
           (64, 5, 60)]


@pytest.mark.parametrize("dl,p,dr", LANCZOS)
@pytest.mark.parametrize("max_iter", [2, 3, 15])
def test_local_krylov_at_the_sizes_where_its_kernels_change(dl, p, dr, max_iter):
    kv = GE.load_package()
    from oracle import tdvp as OT
    from oracle.blocksparse import Tensor as OTensor
    rng = np.random.default_rng([dl, p, dr])
    print(f"case local_krylov {dl}x{p}x{dr} max_iter {max_iter}", flush=True)

    def herm(n):
        g = cplx(rng, n, n)
        return (g + g.conj().T) / np.sqrt(8.0 * n)

    # one charge sector: H = h_L + h_s + h_R over channels (not begun, done)
    L, R = np.zeros((dl, 2, dl), complex), np.zeros((dr, 2, dr), complex)
    L[:, 0], L[:, 1] = np.eye(dl), herm(dl)
    R[:, 1], R[:, 0] = np.eye(dr), herm(dr)
    W = np.zeros((p, 2, p, 2), complex)
    W[:, 0, :, 0] = W[:, 1, :, 1] = np.eye(p)
    W[:, 0, :, 1] = herm(p)
    x = cplx(rng, dl, p, dr)
    parts = [((1, -1, -1), {(0, 0, 0): L}), ((1, 1, -1, -1), {(0, 0, 0, 0): W}), ((-1, 1, 1), {(0, 0, 0): R}),
             ((1, 1, -1), {(0, 0, 0): x})]
    tl, tw, tr, tx = (kv.Tensor.from_blocks(d, b) for d, b in parts)
    ol, ow, orr, ox = (OTensor(d, b) for d, b in parts)
    for reverse in (False, True):
        want, info = OT.local_krylov(ol, ox, ow, None, orr, 0.1, 1e-8, max_iter, reverse, 1)
        got, ex = kv.local_krylov(tl, kv.transpose(tx, range(3)), tw, None, tr, 0.1, 1e-8, max_iter, reverse=reverse)
        (g,), (w,) = got.to_blocks()[1].values(), want.blocks.values()
        # both sides: at most 15 Krylov vectors of rounding errors against a unit vector
        assert np.linalg.norm(g - w) < 1e-12
        assert ex["iters"] == info.iters and ex["converged"] == info.converged


# the Jacobi route's row-count variants (64, 256, 512, more), square, wide and tall, one row or
# column, odd widths, the widest it takes and the largest matrix; sectors share one launch
SVD = [[(1, 1)], [(1, 9), (9, 1), (2, 3)], [(33, 32), (5, 64), (63, 64)], [(63, 63), (64, 17), (256, 31)],
       [(1, 128), (200, 63), (256, 2)], [(257, 12), (40, 512)], [(513, 33), (3, 1500)], [(4161, 63)], [(63, 4161)]]
SPECTRA = {"flat": lambda k: np.linspace(1.0, 0.5, k), "graded": lambda k: 10.0 ** -np.linspace(0, 14, k),
           "repeated": lambda k: np.where(np.arange(k) < (k + 1) // 2, 1.0, 1e-3),
           "deficient": lambda k: np.where(np.arange(k) < (k + 1) // 2, 1.0 / (1 + np.arange(k)), 0.0)}


@pytest.mark.parametrize("shapes", SVD)
@pytest.mark.parametrize("spectrum", [*SPECTRA, "copies"])
@pytest.mark.parametrize("l2r", [True, False])
def test_small_sectors_svd(shapes, spectrum, l2r):
    kv = GE.load_package()
    rng = np.random.default_rng([len(shapes), *shapes[0]])
    print(f"case svd {shapes} {spectrum} l2r {l2r}", flush=True)

    def unitary(m, k):
        return np.linalg.qr(cplx(rng, m, k))[0]

    blocks = {}
    for q, (m, n) in enumerate(shapes):
        k = min(m, n)
        if spectrum == "copies":  # equal rows and columns, many of them zero
            a = cplx(rng, m, n)
            a[k // 2:], a[:, k // 3 + 1:] = 0, a[:, :1]
            blocks[(q, q)] = a
            continue
        blocks[(q, q)] = (unitary(m, k) * SPECTRA[spectrum](k)) @ unitary(n, k).conj().T
    t = kv.Tensor.from_blocks((1, -1), blocks)
    # with a truncating cutoff the route starts at a longer side of 128
    cutoffs = [-1.0] if min(map(max, shapes)) < 128 else [1e-13 if spectrum in ("deficient", "copies") else 0.0, -1.0]
    for cutoff in cutoffs:
        left, right = kv.svd_impl(t, 1, cutoff, 10 ** 6, l2r)
        L, R = left.to_blocks()[1], right.to_blocks()[1]
        for q, (m, n) in enumerate(shapes):
            M = blocks[(q, q)]
            if (q, q) not in L:  # nothing of the sector is above the cutoff
                assert np.linalg.norm(M, 2) <= 1e-13
                continue
            u, v = L[(q, q)], R[(q, q)]
            iso = u.conj().T @ u if l2r else v @ v.conj().T
            k = min(m, n)
            assert cutoff >= 0 or iso.shape == (k, k)
            # k rotations or reflections over a side of max(m, n), a few roundings each
            tol = 40 * EPS * np.sqrt(k * max(m, n))
            assert np.abs(iso - np.eye(len(iso))).max() < tol
            assert np.linalg.norm(u @ v - M) <= tol * np.linalg.norm(M) + (cutoff if cutoff > 0 else 0) * k
            s = np.sort(np.linalg.norm(v, axis=1) if l2r else np.linalg.norm(u, axis=0))[::-1]
            want = np.linalg.svd(M, compute_uv=False)[:len(s)]
            assert np.abs(s - want).max() <= tol * want[0]


def test_svd_of_a_non_finite_sector_is_refused():
    kv = GE.load_package()
    m = np.ones((128, 3), complex)
    m[2, 1] = np.nan
    with pytest.raises(kv.KVError):
        kv.svd_impl(kv.Tensor.from_blocks((1, -1), {(0, 0): m}), 1, 1e-10, 10, True)


# sides of the eigenvectors' back-transformation: its variants' limits (64, 128, 256, 512) and
# one more, kept counts that its columns per wave do not divide, sectors of different sides
GRAM = [([64], 63), ([65, 65], 130), ([127], 31), ([128, 129], 100), ([256], 255), ([257, 70], 33), ([511], 7), ([513], 200)]


@pytest.mark.parametrize("sides,keep", GRAM)
@pytest.mark.parametrize("l2r", [True, False])
def test_gram_sectors_svd(sides, keep, l2r, monkeypatch):
    monkeypatch.setenv("KV_SVD", "full")  # not the block subspace route
    kv = GE.load_package()
    rng = np.random.default_rng(sides)
    print(f"case gram svd {sides} keep {keep} l2r {l2r}", flush=True)
    blocks = {}
    for q, n in enumerate(sides):
        u, v = np.linalg.qr(cplx(rng, n, n))[0], np.linalg.qr(cplx(rng, n + 5, n))[0]
        m = (u * 10.0 ** (-2.0 * (np.arange(n) + 0.1 * q) / n)) @ v.conj().T
        blocks[(q, q)] = m if l2r else m.conj().T
    left, right = kv.svd_impl(kv.Tensor.from_blocks((1, -1), blocks), 1, 1e-10, keep, l2r)
    L, R = left.to_blocks()[1], right.to_blocks()[1]
    assert sum(b.shape[1] for b in L.values()) == min(keep, sum(sides))
    for q, n in enumerate(sides):
        u, v = L[(q, q)], R[(q, q)]
        k = u.shape[1]
        U, s, V = np.linalg.svd(blocks[(q, q)], full_matrices=False)
        iso = u.conj().T @ u if l2r else v @ v.conj().T
        # n reflectors and as many merges of orthonormal bases, a few roundings each; the kept
        # subspace turns by the Gram matrix's rounding over the gap of its values at the cut
        assert np.abs(iso - np.eye(k)).max() < 16 * n * EPS
        gap = s[k - 1] ** 2 - (s[k] ** 2 if k < n else 0.0)
        assert np.linalg.norm(u @ v - (U[:, :k] * s[:k]) @ V[:k]) < 64 * n * EPS / gap


# sides around the merges (8, 16, ... 256) of the tridiagonal divide and conquer and its largest, and
# around the side (128) whose reduction stays in registers;
# spectra whose values deflate in part, all at once and not at all
@pytest.mark.parametrize("sides", [[128], [65, 64], [127, 66], [129], [130, 66], [97, 160, 95], [193], [256], [384, 64], [512, 65]])
@pytest.mark.parametrize("spectrum", ["equal", "steps", "deficient", "graded"])
def test_gram_sectors_of_clustered_values(sides, spectrum, monkeypatch):
    monkeypatch.setenv("KV_SVD", "full")
    kv = GE.load_package()
    rng = np.random.default_rng([*sides, len(spectrum)])
    print(f"case clustered gram {sides} {spectrum}", flush=True)
    blocks, rank = {}, 0
    for q, n in enumerate(sides):
        u, v = np.linalg.qr(cplx(rng, n, n))[0], np.linalg.qr(cplx(rng, n + 3, n))[0]
        x = np.arange(n) / n
        s = {"equal": 0 * x + 1, "steps": 0.5 ** np.floor(4 * x), "deficient": np.where(x < 0.5, 1 - x, 0.0),
             "graded": 10.0 ** (-3.0 * x)}[spectrum]
        rank += np.count_nonzero(s)
        blocks[(q, q)] = (u * s) @ v.conj().T
    left, right = kv.svd_impl(kv.Tensor.from_blocks((1, -1), blocks), 1, 1e-6, rank, True)
    L, R = left.to_blocks()[1], right.to_blocks()[1]
    assert sum(b.shape[1] for b in L.values()) == rank
    for (q, _), m in blocks.items():
        n, u = m.shape[0], L[(q, q)]
        # as in test_gram_sectors_svd; nothing is cut off but zeros, so all of m comes back
        assert np.abs(u.conj().T @ u - np.eye(u.shape[1])).max() < 16 * n * EPS
        assert np.linalg.norm(u @ R[(q, q)] - m) < 64 * n * EPS
