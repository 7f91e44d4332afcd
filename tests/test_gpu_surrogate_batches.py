"""Batch sizes of the surrogate step at its edges: one cell, remainders of 16-
and 64-cell groups, both sides of the switch between 16 and 64 cells a wave,
and rejected cells in one run (a workgroup's list longer than its waves).

Rejected cells anywhere: none, all, one run, one a workgroup's first or last
cell; and their cost, which does not depend on where they lie.

A cell's result does not depend on its batch: the network's sums run in one
order in every variant and a rejected cell takes the plain step, so equality
is exact."""
import time

import numpy as np
import pytest

from openstc_amd import _lib as L
from openstc_amd import surrogate as S
from test_gpu_surrogate import env  # noqa: F401  (fixture)

pytestmark = pytest.mark.gpu
BIG = 64 * 12 * 256 // 2 + 17  # past the switch on 256 CUs


@pytest.fixture(scope="module")
def batch(env):  # noqa: F811
    ctx = env[0]
    m = np.load(S.DEFAULT_WEIGHTS, allow_pickle=False)
    sur = S.Surrogate.load(ctx)
    t, p, y, dt = (np.ascontiguousarray(np.resize(m["heldout_" + k], (BIG,) + m["heldout_" + k].shape[1:]))
                   for k in ("t", "p", "y", "dt"))
    t[3000:5500] = 5000.0  # one run outside the trained range
    dev = [S.DeviceArray(a) for a in (t, p, y, dt)]
    out = S.DeviceArray(nbytes=BIG * 9 * 8)
    st = sur.step(BIG, *(a.p for a in dev), out.p)
    got = out.get(np.float64, (BIG, 9))
    yield sur, dev, out, got, st, S.plain_step(ctx, t, p, y, dt)
    for a in dev + [out]:
        a.free()
    sur.close()


def test_rejected_cells_take_the_plain_step(batch):
    _, _, _, got, st, plain = batch
    print("[gpu-sur-n] stats", st, flush=True)
    assert st[0] == BIG and st[1] >= 2500
    assert np.array_equal(got[3000:5500], plain[3000:5500])
    same = np.all(got == plain, axis=1)
    assert same.sum() >= st[1] + st[2] + st[3]


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 1000, 3001, 16385, BIG - 18, BIG - 17, BIG - 1])
def test_size(batch, n):
    sur, dev, out, got, _, _ = batch
    st = sur.step(n, *(a.p for a in dev), out.p)
    print("[gpu-sur-n]", n, st, flush=True)
    assert st[0] == n and 0 <= st[1] + st[2] + st[3] <= n
    assert st[1] >= max(0, min(n, 5500) - 3000)
    assert np.array_equal(out.get(np.float64, (BIG, 9))[:n], got[:n])


def resized(n):
    m = np.load(S.DEFAULT_WEIGHTS, allow_pickle=False)
    return [np.ascontiguousarray(np.resize(m["heldout_" + k], (n,) + m["heldout_" + k].shape[1:]))
            for k in ("t", "p", "y", "dt")]


@pytest.mark.parametrize("n", [1, 64, 16385, 300001])
@pytest.mark.parametrize("where", ["none", "all", "run", "every 97th"])
def test_where_cells_are_rejected(env, n, where):  # noqa: F811
    """Pieces of 64 rejected cells that span many lists, or many pieces of
    one list, more than the device holds at once among them (300 001 of them
    are 4 688 waves)."""
    print("[gpu-sur-n] rejected:", where, "of", n, flush=True)
    ctx = env[0]
    sur = S.Surrogate.load(ctx)
    t, p, y, dt = resized(n)
    keep = t.copy()
    if where == "all":
        t[:] = 5000.0
    elif where == "run":
        t[n // 3:n // 3 + max(1, n // 4)] = 5000.0
    elif where == "every 97th":
        t[::97] = 5000.0
    bad = t != keep
    dev = [S.DeviceArray(a) for a in (t, p, y, dt)]
    out = S.DeviceArray(nbytes=n * 9 * 8)
    st = sur.step(n, *(a.p for a in dev), out.p)
    got, plain = out.get(np.float64, (n, 9)), S.plain_step(ctx, t, p, y, dt)
    print("[gpu-sur-n] stats", st, flush=True)
    assert st[0] == n and st[1] >= bad.sum()
    assert np.array_equal(got[bad], plain[bad])
    assert np.all(got == plain, axis=1).sum() >= st[1] + st[2] + st[3]
    if where == "none":
        accepted = ~np.all(got == plain, axis=1)
        assert accepted.sum() <= n - (st[1] + st[2] + st[3])
    for a in dev + [out]:
        a.free()
    sur.close()


def test_cost_of_a_cluster(env):  # noqa: F811
    """5 % of a batch rejected in one run cost what 5 % spread out cost: the
    plain steps of a run are shared by the whole device (1.3: the batches of
    a list bound to its own waves took 1.65 times as long)."""
    n = 1500000
    ctx = env[0]
    sur = S.Surrogate.load(ctx)
    t, p, y, dt = resized(n)
    spread, run = t.copy(), t.copy()
    spread[::20] = 5000.0
    run[n // 3:n // 3 + n // 20] = 5000.0
    rest, out = [S.DeviceArray(a) for a in (p, y, dt)], S.DeviceArray(nbytes=n * 9 * 8)
    dev = [S.DeviceArray(spread), S.DeviceArray(run)]

    def took(d, reps=20):
        t0 = time.perf_counter()
        for _ in range(reps):
            L.check(ctx.lib.ostc_surrogate_step(sur.h, n, d.p, *(a.p for a in rest), out.p, None, None), "step")
        L.check(ctx.lib.ostc_device_sync(), "sync")
        return (time.perf_counter() - t0) / reps

    for d in dev:
        took(d, 5)
    best = [min(took(d) for _ in range(5)) for d in dev]
    print("[gpu-sur-n] spread %.1f us, one run %.1f us" % tuple(1e6 * b for b in best), flush=True)
    assert best[1] < 1.3 * best[0]
    for a in dev + rest + [out]:
        a.free()
    sur.close()
