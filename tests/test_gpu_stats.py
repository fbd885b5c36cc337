"""The module clocks and the device-time counters of a sweep."""
import os
import sys
import time

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import __graft_entry__ as GE  # noqa: E402

pytestmark = pytest.mark.gpu
MODULES = ("Evl-2", "Evl-1", "Evl-0", "SVD", "Update", "Sweep")


def chain(kv, p, bonds, local, ctx=None):
    """A chain of one charge sector: random sites of p levels between bonds, and H = sum h_i
    (local, a two-channel MPO) or H = h_1 h_2 ... (one channel)."""
    rng = np.random.default_rng([p, *bonds])
    b = [1, *bonds, 1]

    def tensor(dirs, a):
        return kv.Tensor.from_blocks(dirs, {(0,) * a.ndim: a}, ctx)

    mps, mpo = [], []
    for i in range(len(b) - 1):
        s = (b[i], p, b[i + 1])
        mps.append(tensor((1, 1, -1), (rng.standard_normal(s) + 1j * rng.standard_normal(s)) / np.sqrt(np.prod(s))))
        h = np.diag(np.linspace(-1.0, 1.0, p)).astype(complex)
        if not local:
            mpo.append(tensor((1, 1, -1, -1), h[:, None, :, None]))
            continue
        w = np.zeros((p, 2, p, 2), complex)  # channels (not begun, done)
        w[:, 0, :, 0] = w[:, 1, :, 1] = np.eye(p)
        w[:, 0, :, 1] = h
        w = w[:, :1] if i == 0 else w
        mpo.append(tensor((1, 1, -1, -1), w[..., 1:] if i == len(b) - 2 else w))
    return mps, mpo


@pytest.mark.parametrize("step", ["one_site", "two_site"])
def test_update_time_holds_the_environments_device_time(step):
    """The environment updates' launches run on after the call that queues them: their time
    belongs to Update, and to no other module as well."""
    kv = GE.load_package()
    print(f"case module clocks {step}", flush=True)
    eng = kv.TDVP(*chain(kv, 32, (32, 1024, 32), True), cutoff=1e-12, maxdim=1024, dt=0.05, max_iter=3)
    run = getattr(eng, step)
    run()  # tile tuning
    eng.reset_stats()
    t0 = time.perf_counter()
    run()
    wall = time.perf_counter() - t0
    st = eng.stats()
    assert st["env_gpu_s"] > 0
    assert st["Update"] >= st["env_gpu_s"]
    assert all(st[m] >= 0 for m in MODULES)
    assert sum(st[m] for m in MODULES) <= wall

def test_tile_tuning_is_not_booked_on_the_launch_before():
    """A context's first step times the tiles of a product between two launches of a matvec; the
    fold before it must not be charged for that."""
    kv = GE.load_package()
    print("case tuning", flush=True)

    def fold_times():
        ctx = kv.Context(0)  # the tuned tiles are the context's
        # site 2's last product: 900 x 120, K = 120: tuned, and too shallow to be cut into K chunks
        eng = kv.TDVP(*chain(kv, 30, (30, 120, 30), False, ctx), cutoff=1e-12, maxdim=120, dt=0.05, max_iter=2)
        t = []
        for _ in range(2):
            eng.reset_stats()
            eng.one_site()
            t.append(eng.stats()["heff_wfold_gpu_s"])
        del eng
        ctx.close()
        return t

    fold_times()  # loads the kernels
    pairs = [fold_times() for _ in range(3)]
    first, second = (min(p[k] for p in pairs) for k in (0, 1))
    assert 0 < first < 3 * second, pairs
