"""The strash by level sweeps and hashing rounds against the wave sweep and the
oracle on what it takes by size: whole graphs of any size, one that holds the
same deep logic twice (more rounds than are tried, so it gives way), rewrites
of more than 1,024 objects per level, and batches on both sides of 64 times
their largest member."""
import sys

import numpy as np
import pytest

import culs_amd
import oracle_ffi as O

pytestmark = pytest.mark.gpu


def same(a, b):
    return all(np.array_equal(np.asarray(x), np.asarray(y)) for x, y in zip(a, b))


def log(*a):
    print(*a)
    sys.stdout.flush()


def twice(nPIs, f0, f1, pos):
    """The ANDs of a graph twice over the same PIs: every node of the second copy
    is a duplicate, found level by level."""
    n, first = len(f0), nPIs + 1

    def copy(x):
        x = np.asarray(x, np.uint32)
        return np.where(x >> 1 >= first, x + 2 * (n - first), x).astype(np.uint32)

    return (nPIs, np.concatenate([f0, copy(f0[first:])]), np.concatenate([f1, copy(f1[first:])]),
            np.concatenate([pos, copy(pos)]))


GRAPHS = [
    ("one_and", lambda c: (2, np.array([0, 0, 0, 2], np.uint32), np.array([0, 0, 0, 5], np.uint32),
                           np.array([6], np.uint32))),
    ("random_500", lambda c: c.gen_random(20, 500, 8, 100, 1).arrays()),
    ("random_20k", lambda c: c.gen_random(64, 20000, 32, 1000, 1).arrays()),
    ("wide_60k", lambda c: c.gen_random(512, 60000, 100, 20000, 2).arrays()),
    ("mult8_twice", lambda c: twice(*c.gen_multiplier(8, 0.1, 2).arrays())),
    ("mult32_twice", lambda c: twice(*c.gen_multiplier(32, 0.1, 2).arrays())),
]


@pytest.mark.parametrize("name,make", GRAPHS, ids=[g[0] for g in GRAPHS])
def test_strash_of_raw_graphs(gpu_ctx, name, make):
    log("strash routes:", name)
    g = make(gpu_ctx)
    want, depth = O.strash(*g)
    for schedule in (0, culs_amd.GLS_ST_WAVES, culs_amd.GLS_ST_LEVELS):
        a = gpu_ctx.from_arrays(*g).strash(schedule=schedule)
        log(name, schedule, "final_strash", a.last_op()["final_strash"], "rounds", a.last_op()["strash_rounds"])
        assert same(a.arrays(), want) and a.stats().levels == depth, schedule
        if schedule == 0:
            assert a.last_op()["final_strash"] == (2 if name.endswith("twice") else 1)


@pytest.mark.parametrize("pis,ands,window", [(512, 60000, 20000), (64, 30000, 8000)])
@pytest.mark.parametrize("zeros", [False, True])
def test_rewrite_of_wide_graphs(gpu_ctx, pis, ands, window, zeros):
    log("wide rewrite:", pis, ands, window, zeros)
    a = gpu_ctx.gen_random(pis, ands, 100, window, 3).strash()
    b, x = a.copy(), a.arrays()
    a.rewrite(use_zeros=zeros)
    assert a.last_op()["final_strash"] == 1
    b.rewrite(use_zeros=zeros, full_strash=True)
    assert same(a.arrays(), b.arrays()) and a.stats().levels == b.stats().levels
    assert same(a.arrays(), O.rw(*x, use_zeros=zeros)[0])


@pytest.mark.parametrize("count", [1, 2, 63, 64, 66])
@pytest.mark.parametrize("double", [False, True])
def test_batches_around_the_line(gpu_ctx, count, double):
    log("batched strash:", count, double)
    graphs = [gpu_ctx.gen_random(20, 300, 8, 100, 40 + i).arrays() for i in range(count)]
    if double:
        graphs[0] = twice(*gpu_ctx.gen_multiplier(8, 0.1, 2).arrays())
    aigs = [gpu_ctx.from_arrays(*g) for g in graphs]
    gpu_ctx.batch_strash(aigs)
    for a, g in zip(aigs, graphs):
        want, depth = O.strash(*g)
        assert same(a.arrays(), want) and a.stats().levels == depth
