"""H_eff in FP32 and split BF16 where its products are cut into K chunks."""
import os
import subprocess
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import __graft_entry__ as GE  # noqa: E402
from oracle import tdvp as T  # noqa: E402
from oracle.blocksparse import Tensor as OT  # noqa: E402

pytestmark = pytest.mark.gpu


def operands(dl, p, dr, w):
    """L, x, W, R of one site in one charge sector; the products' K are dl and w dr."""
    rng = np.random.default_rng([dl, p, dr, w])

    def cplx(*s):
        return rng.standard_normal(s) + 1j * rng.standard_normal(s)

    W = np.zeros((p, w, p, w), complex)
    W[np.arange(p)[:, None], np.arange(w), np.arange(p)[:, None], np.arange(w)] = cplx(p, w)
    return (((1, -1, -1), cplx(dl, w, dl)), ((1, 1, -1), cplx(dl, p, dr)), ((1, 1, -1, -1), W),
            ((-1, 1, 1), cplx(dr, w, dr)))


def both(kv, ops):
    return ([kv.Tensor.from_blocks(d, {(0,) * a.ndim: a}) for d, a in ops],
            [OT(d, {(0,) * a.ndim: a}) for d, a in ops])


def launched():
    """Kernels of one split-BF16 H_eff as torch's profiler lists them, in a process of its own: torch
    finds the GPU only where it is loaded before the engine."""
    from torch.profiler import ProfilerActivity, profile
    kv = GE.load_package()
    (L, x, W, R), _ = both(kv, PINNED)
    with profile(activities=[ProfilerActivity.CUDA]) as prof:
        kv.apply_single(L, x, W, R, "bf16x3")
    for e in prof.key_averages():
        print(e.key, flush=True)


PINNED = operands(257, 1, 300, 2)


@pytest.mark.parametrize("tile", ["64", "128"])
def test_pinned_tile_runs_in_plans_cut_into_chunks(tile, monkeypatch):
    """KV_SPLIT_TILE names the split-BF16 kernel that runs, with 4 and 8 K chunks."""
    kv = GE.load_package()
    monkeypatch.setenv("KV_SPLIT_TILE", tile)
    print(f"case pinned tile {tile}", flush=True)
    run = subprocess.run([sys.executable, os.path.abspath(__file__)], capture_output=True, text=True, timeout=100)
    assert run.returncode == 0, run.stderr
    names = run.stdout.splitlines()
    gemm = [n for n in names if "zgemm" in n]
    assert any("sum_parts" in n for n in names)
    assert len(gemm) == 2 and all(f", {tile}, {tile}, " in n for n in gemm), gemm
    (L, x, W, R), ref = both(kv, PINNED)
    (got,) = kv.apply_single(L, x, W, R, "bf16x3").to_blocks()[1].values()
    (want,) = T.apply_single(*ref).blocks.values()
    # split BF16 as in test_gpu_parity: about 3 * 2^-18 of |a||b| per product, over the two stages
    (mag,) = T.apply_single(*(OT(t.dirs, {q: abs(b).astype(complex) for q, b in t.blocks.items()})
                              for t in ref)).blocks.values()
    assert abs(got - want).max() <= 2e-4 * mag.real.max()


# (Dl, levels, Dr, W's channels): K of the two products 127 (uncut), 128 and 129 (two chunks), 255 and
# 256 (two and four), 1047 and 2094 (16 and 32 chunks, of which the last two are empty), many tiles
CHUNKS = [(127, 1, 127, 1), (128, 1, 128, 1), (129, 3, 65, 2), (255, 2, 256, 1), (1047, 1, 3, 1), (5, 1, 1047, 2),
          (600, 1, 520, 1)]


@pytest.mark.parametrize("dl,p,dr,w", CHUNKS)
@pytest.mark.parametrize("precision", ["fp32", "bf16x3"])
def test_heff_at_the_chunk_limits(dl, p, dr, w, precision):
    kv = GE.load_package()
    print(f"case chunks {dl}x{p}x{dr} w {w} {precision}", flush=True)
    (L, x, W, R), ref = both(kv, operands(dl, p, dr, w))
    (got,) = kv.apply_single(L, x, W, R, precision).to_blocks()[1].values()
    (want,) = T.apply_single(*ref).blocks.values()
    (mag,) = T.apply_single(*(OT(t.dirs, {q: abs(b).astype(complex) for q, b in t.blocks.items()})
                              for t in ref)).blocks.values()
    # two products in FP32: a rounding per term and a few for the operands, the fold and the complex
    # products' three real ones, in units of the products of absolute values; split BF16 also drops
    # 3 * 2^-18 of each of a complex product's four real ones, in either product
    tol = 4 * (dl + w * dr + 16) * 2.0 ** -24 + (24 * 2.0 ** -18 if precision == "bf16x3" else 0)
    assert np.all(abs(got - want) <= tol * mag.real)


if __name__ == "__main__":
    launched()
