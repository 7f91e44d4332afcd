"""Batch sizes of the surrogate step at its edges: one cell, remainders of 16-
and 64-cell groups, both sides of the switch between 16 and 64 cells a wave,
and rejected cells in one run (a workgroup's list longer than its waves).

A cell's result does not depend on its batch: the network's sums run in one
order in every variant and a rejected cell takes the plain step, so equality
is exact."""
import numpy as np
import pytest

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
