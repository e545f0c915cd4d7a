"""Evaluation of every node against the oracle, bit for bit, where a wavefront
is partly filled: counts of ANDs around its two or eight nodes and around the
count (49152) at which eight follow two."""
import sys

import numpy as np
import pytest

import oracle_ffi as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ands", [1, 2, 3, 7, 8, 9, 49151, 49152, 49153, 49157])
@pytest.mark.parametrize("pis,window", [(12, 300), (64, 5000)])
def test_evaluate_counts(gpu_ctx, ands, pis, window):
    print("evaluate %d ANDs, %d PIs, window %d" % (ands, pis, window))
    sys.stdout.flush()
    nPIs, f0, f1, _ = gpu_ctx.gen_random(pis, 80000 if ands > 9 else 200, 40, window, 21).strash().arrays()
    n = nPIs + 1 + ands
    assert len(f0) >= n
    # the first ands ANDs, each without fanout a PO
    f0, f1 = f0[:n], f1[:n]
    used = np.zeros(n, bool)
    used[f0[nPIs + 1:] >> 1] = used[f1[nPIs + 1:] >> 1] = True
    pos = (2 * np.nonzero(~used[nPIs + 1:])[0] + 2 * (nPIs + 1)).astype(np.uint32)
    a = gpu_ctx.from_arrays(nPIs, f0, f1, pos).strash()
    assert len(a.arrays()[1]) == n
    a.reorder()
    r = a.arrays()
    want = O.cuts(*r)
    for z in (False, True):
        assert np.array_equal(a.evaluate(use_zeros=z), O.evaluate(*r, want, use_zeros=z)), z
