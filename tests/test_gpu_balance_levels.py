"""Balance at the sizes where a level stops fitting the workgroup that rebuilds
it in LDS (2048 covers, 4096 inputs, 3072 possible ANDs), bit for bit against
the oracle: a single graph, and as a member of a batch beside small ones."""
import sys

import numpy as np
import pytest

import oracle_ffi as O

pytestmark = pytest.mark.gpu


def same(a, b):
    return all(np.array_equal(np.asarray(x), np.asarray(y)) for x, y in zip(a, b))


def layered(layers, nPIs, seed):
    """layers of (covers, inputs): each cover a chain of ANDs over complemented
    covers of the layer below (the first: PIs of either polarity); the last
    layer drives the POs, so some covers below are not reached.  Few PIs make
    equal pairs, repeated inputs and constant covers."""
    rng = np.random.default_rng(seed)
    f0, f1 = [0] * (nPIs + 1), [0] * (nPIs + 1)
    below = None
    for covers, k in layers:
        tops = []
        for _ in range(covers):
            if below is None:
                lits = 2 * rng.integers(1, nPIs + 1, k) + rng.integers(0, 2, k)
            else:
                lits = rng.choice(below, k) + 1
            cur = int(lits[0])
            for x in lits[1:]:
                f0.append(cur)
                f1.append(int(x))
                cur = 2 * (len(f0) - 1)
            tops.append(cur)
        below = np.array(tops)
    return nPIs, np.array(f0, np.uint32), np.array(f1, np.uint32), below.astype(np.uint32)


SHAPES = [
    [(1, 2)],
    [(2047, 2)], [(2048, 2)], [(2049, 2)],            # covers, and inputs at 4096
    [(1365, 3)], [(1366, 3)],                         # inputs 4095 and 4098
    [(1024, 4)], [(768, 5)], [(769, 5)], [(512, 8)],  # possible ANDs 3072, 3072, 3076, 3584
    [(9000, 2), (40, 3)],                             # a frontier of more than 8192
    [(300, 3), (3000, 3), (200, 6), (64, 40), (2049, 2), (65, 3)],   # both kinds of level
]


@pytest.mark.parametrize("shape", SHAPES, ids=["-".join("%dx%d" % s for s in x) for x in SHAPES])
def test_balance_levels_at_the_limits(gpu_ctx, shape):
    print("balance levels:", shape)
    sys.stdout.flush()
    # few PIs and many: with many, nearly every AND is a new node
    for nPIs in (12, 5000):
        g = layered(shape, nPIs, 5)
        a = gpu_ctx.from_arrays(*g)
        a.balance(update_level=False)
        assert same(a.arrays(), O.balance(*g)), nPIs


@pytest.mark.parametrize("shape", [SHAPES[2], SHAPES[3], SHAPES[-1]], ids=["fits", "wide", "mixed"])
def test_batch_balance_levels_at_the_limits(gpu_ctx, shape):
    print("batch balance levels:", shape)
    sys.stdout.flush()
    graphs = [layered([(50, 3), (20, 4)], 30, 1), layered(shape, 5000, 2), layered([(7, 2)], 9, 3)]
    aigs = [gpu_ctx.from_arrays(*g) for g in graphs]
    gpu_ctx.batch_balance(aigs, update_level=False)
    for a, g in zip(aigs, graphs):
        assert same(a.arrays(), O.balance(*g))


RAW_SHUFFLE = pytest.mark.xfail(strict=True, reason="`b -s` of a graph whose fanins are not in strashed order: the "
                                "order in which a cover's inputs are shuffled differs from the oracle's")


@pytest.mark.parametrize("covers,k", [(40, 6), (1024, 4), (300, 11)])
@pytest.mark.parametrize("shuffle,strashed", [(False, False), (False, True), (True, True),
                                              pytest.param(True, False, marks=RAW_SHUFFLE)])
def test_balance_pairs_that_exist(gpu_ctx, covers, k, shuffle, strashed):
    """Covers over PIs whose pairs the levels before have created: few of them
    (found nodes put back meet older ones), and more than a level has room for."""
    print("balance existing pairs: %d covers of %d inputs, shuffle %s" % (covers, k, shuffle))
    sys.stdout.flush()
    rng = np.random.default_rng(k)
    nPIs = 9
    f0, f1, pos = [0] * (nPIs + 1), [0] * (nPIs + 1), []

    def chain(lits):
        cur = int(lits[0])
        for x in lits[1:]:
            f0.append(cur)
            f1.append(int(x))
            cur = 2 * (len(f0) - 1)
        return cur

    def pis(n):
        return 2 * (1 + rng.permutation(nPIs)[:n]) + rng.integers(0, 2, n)

    below = [chain(pis(rng.integers(2, 5))) for _ in range(200)]
    above = [chain(np.append(pis(rng.integers(2, 4)), x + 1)) for x in below]
    for i in range(covers):
        pos.append(chain(np.append(pis(min(k - 1, nPIs)), above[i % len(above)] + 1)))
    g = nPIs, np.array(f0, np.uint32), np.array(f1, np.uint32), np.array(pos, np.uint32)
    a = gpu_ctx.from_arrays(*g)
    if strashed:
        g = a.strash().arrays()
    a.balance(update_level=False, shuffle=shuffle)
    assert same(a.arrays(), O.balance(*g, sort_dec_id=0 if shuffle else 1))
