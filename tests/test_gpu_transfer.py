"""Arrays fetched from the device: sizes around the staging (2 MiB in all) and
its pieces (4 MiB of an array), both literal conventions, arrays left out,
repeated and after a copy.  A strashed level-major AIG strashes to itself, so
the arrays are known without the device."""
import sys

import numpy as np
import pytest

import culs_amd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def base(gpu_ctx):
    return {"small": gpu_ctx.gen_random(64, 300000, 32, 1000, 1).strash().arrays(),
            "large": gpu_ctx.gen_random(256, 1500000, 32, 2000, 1).strash().arrays()}


def prefix(g, n, n_pos):
    """The first n objects; every AND without fanout a PO, filled up to n_pos."""
    nPIs, f0, f1, _ = g
    assert len(f0) >= n
    f0, f1 = f0[:n], f1[:n]
    used = np.zeros(n, bool)
    used[f0[nPIs + 1:] >> 1] = used[f1[nPIs + 1:] >> 1] = True
    pos = 2 * (np.nonzero(~used[nPIs + 1:])[0] + nPIs + 1)
    if n_pos is not None:
        assert len(pos) <= n_pos
        pos = np.concatenate([pos, np.arange(n_pos - len(pos)) % 4])
    return nPIs, f0, f1, pos.astype(np.uint32)


def fetch(a, conv, want):
    out = [np.full(len(w), 77, np.uint32) for w in want]
    ptr = [o.ctypes.data if len(o) else None for o in out]
    a.ctx.check(culs_amd.lib().gls_aig_to_arrays(a._h, *ptr, conv), "gls_aig_to_arrays")
    return out


SIZES = [("small", 200, None), ("small", 180000, 524287 - 360000), ("small", 180000, 524288 - 360000),
         ("small", 180000, 524289 - 360000), ("large", 1048575, None), ("large", 1048576, None),
         ("large", 1048577, None)]


@pytest.mark.parametrize("which,n,n_pos", SIZES)
def test_fetched_arrays(gpu_ctx, base, which, n, n_pos):
    print("fetch: %d objects, POs %s" % (n, n_pos))
    sys.stdout.flush()
    g = prefix(base[which], n, n_pos)
    for conv in (0, 1):
        want = [np.where(x < 2, 1 - x.astype(np.int64), x).astype(np.uint32) if conv else x for x in g[1:]]
        if conv:
            want[0][:g[0] + 1] = want[1][:g[0] + 1] = 0
        a = gpu_ctx.from_arrays(*g).strash()
        assert a.stats().on_device == 1
        b = a.copy()
        for x, times in ((a, 3), (b, 1)):
            for _ in range(times):
                assert all(np.array_equal(p, q) for p, q in zip(fetch(x, conv, want), want))
                assert x.stats().on_device == 0
        c = a.copy().strash()
        a.ctx.check(culs_amd.lib().gls_aig_to_arrays(c._h, None, None, None, conv), "gls_aig_to_arrays")
        assert all(np.array_equal(p, q) for p, q in zip(fetch(c, conv, want), want))
