"""Simulation where fanins lie just inside and outside the values kept on chip
(4,096 ids, of which 3,072 below a chunk of 1,024), against the oracle."""
import sys

import numpy as np
import pytest

import oracle_ffi as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nPIs", [1, 5, 1030, 4100])
@pytest.mark.parametrize("dist", [1, 63, 64, 1023, 1024, 1025, 3071, 3072, 3073, 4095, 4096, 4097, 6000])
def test_simulate_fanin_distances(gpu_ctx, nPIs, dist):
    print("simulate: %d PIs, fanins %d ids back" % (nPIs, dist))
    sys.stdout.flush()
    rng = np.random.default_rng(dist)
    n = nPIs + 1 + 9000
    ids = np.arange(nPIs + 1, n)
    # one fanin dist ids back (a PI if that is not an AND), the other nearby
    f0, f1 = np.zeros(n, np.uint32), np.zeros(n, np.uint32)
    back = ids - dist
    a = np.where(back > nPIs, back, 1 + ids % nPIs)
    b = np.maximum(ids - rng.integers(1, 2000, len(ids)), 1)
    f0[ids], f1[ids] = 2 * a + rng.integers(0, 2, len(ids)), 2 * b + rng.integers(0, 2, len(ids))
    pos = (2 * ids[::7] + 1).astype(np.uint32)
    g = (nPIs, f0, f1, pos)
    got = gpu_ctx.from_arrays(*g).simulate(2, seed=3)
    assert np.array_equal(got, O.sim_po_words(g, 2, seed=3))
