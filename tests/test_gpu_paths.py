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
