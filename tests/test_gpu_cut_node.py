"""Cut sets of nodes with many candidate pairs, against the oracle bit for bit.

Random AIGs over very few inputs make what the insertion of candidates can
meet: more pairs than one batch of the kernel holds, cuts that contain one
another, tables that lose variables down to constants, and full slot sets that
evict; wide-windowed ones make the candidates that mostly fail to merge."""
import sys

import numpy as np
import pytest

import oracle_ffi as O

pytestmark = pytest.mark.gpu


def pairs_passing(f0, f1, nPIs, cuts):
    """Candidate pairs per AND: pairs of fanin cuts with at most four signature bits."""
    c = np.asarray(cuts).reshape(-1, 8, 5)
    n, used = (c[:, :, 4] >> 27) & 7, (c[:, :, 4] >> 30) & 1
    sig = np.zeros(c.shape[:2], np.uint32)
    for i in range(4):
        sig |= np.where(i < n, np.uint32(1) << (c[:, :, i] & 31), 0).astype(np.uint32)
    ids = np.arange(nPIs + 1, len(f0))
    a, b = f0[ids] >> 1, f1[ids] >> 1
    x = (sig[a][:, :, None] | sig[b][:, None, :]).reshape(len(ids), 64)
    bits = np.unpackbits(x.view(np.uint8).reshape(len(ids), 64, 4), axis=2).sum(axis=2)
    both = (used[a][:, :, None] & used[b][:, None, :]).reshape(len(ids), 64)
    return ((bits <= 4) & (both == 1)).sum(axis=1)


CASES = [(5, 400, 6, 11), (6, 1500, 8, 12), (8, 1500, 12, 13), (10, 1500, 20, 14), (16, 1500, 40, 15),
         (64, 3000, 400, 16)]


@pytest.mark.parametrize("pis,ands,window,seed", CASES)
def test_cut_sets_of_dense_graphs(gpu_ctx, pis, ands, window, seed):
    import culs_amd
    print("cut node: %d PIs, %d ANDs, window %d" % (pis, ands, window))
    sys.stdout.flush()
    a = gpu_ctx.gen_random(pis, ands, 40, window, seed).strash()
    a.reorder()
    nPIs, f0, f1, pos = a.arrays()
    want = O.cuts(nPIs, f0, f1, pos)
    assert pairs_passing(f0, f1, nPIs, want).max() >= 16
    meta = np.asarray(want).reshape(-1, 8, 5)[:, :, 4]
    assert np.any(((meta >> 30) & 1 == 1) & ((meta >> 27) & 7 == 0))       # a constant cut
    for mode in (0, culs_amd.GLS_RW_LEVEL_CUTS, culs_amd.GLS_RW_DATAFLOW_CUTS):
        assert np.array_equal(a.enumerate_cuts(mode), np.asarray(want).reshape(-1)), mode
