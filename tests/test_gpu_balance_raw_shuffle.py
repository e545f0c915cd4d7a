"""`b -s` of graphs that were not strashed: the shuffle takes a cover's inputs in
the order in which the handle's fanins give them (a handle holds each AND's
fanins in ascending order), bit for bit against the oracle on these arrays."""
import sys

import numpy as np
import pytest

import oracle_ffi as O

pytestmark = pytest.mark.gpu


def same(a, b):
    return all(np.array_equal(np.asarray(x), np.asarray(y)) for x, y in zip(a, b))


def graphs(ctx):
    yield "random", ctx.gen_random(40, 4000, 60, 300, 7).arrays()
    yield "multiplier", ctx.gen_multiplier(12, 0.2, 3).arrays()
    for covers, k in ((40, 6), (1024, 4), (300, 11)):
        # covers of k PIs or complemented covers, the fanins in any order
        rng = np.random.default_rng(k)
        nPIs, f0, f1, tops = 9, [0] * 10, [0] * 10, []
        for _ in range(covers):
            lits = 2 * rng.integers(1, nPIs + 1, k) + rng.integers(0, 2, k)
            for j in range(k):
                if tops and rng.random() < 0.3:
                    lits[j] = rng.choice(tops) + 1
            cur = int(lits[0])
            for x in lits[1:]:
                pair = [cur, int(x)]
                rng.shuffle(pair)
                f0.append(pair[0])
                f1.append(pair[1])
                cur = 2 * (len(f0) - 1)
            tops.append(cur)
        yield "covers-%dx%d" % (covers, k), (nPIs, np.array(f0, np.uint32), np.array(f1, np.uint32),
                                             np.array(tops, np.uint32))


def test_shuffle_of_raw_graphs(gpu_ctx):
    for name, g in graphs(gpu_ctx):
        print("b -s, not strashed:", name)
        sys.stdout.flush()
        a = gpu_ctx.from_arrays(*g)
        held = a.arrays()
        assert np.all(held[1] <= held[2]) and same(held[3], g[3])
        a.balance(update_level=False, shuffle=True)
        assert same(a.arrays(), O.balance(*held, sort_dec_id=0)), name
