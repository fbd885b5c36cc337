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
