"""Strash of whole graphs by classes of equal ANDs: graphs in which nodes merge
over several rounds, fold to literals of either polarity and to constants, and
whose class has its lowest wave at another node than its least id; array for
array against the oracle, alone and in a batch."""
import sys

import numpy as np
import pytest

import culs_amd
import oracle_ffi as O

pytestmark = pytest.mark.gpu


def same(a, b):
    return all(np.array_equal(np.asarray(x), np.asarray(y)) for x, y in zip(a, b))


def redundant(nPIs, ands, window, fold, again, seed):
    """Random ANDs over the last `window` objects; a share `fold` of them with a
    constant or their own fanin (complemented or not) as second fanin, a share
    `again` a copy of an earlier one with each fanin behind a folding AND, so
    that its wave is higher until that folds (or, where the copied one is behind
    such ANDs itself, lower)."""
    rng = np.random.default_rng(seed)
    f0, f1 = [0] * (nPIs + 1), [0] * (nPIs + 1)

    def add(a, b):
        f0.append(int(a))
        f1.append(int(b))
        return 2 * (len(f0) - 1)

    while len(f0) < nPIs + 1 + ands:
        n = len(f0)
        kind = rng.random()
        if kind < again and n > nPIs + 4:
            v = int(rng.integers(nPIs + 1, n))
            a, b = f0[v], f1[v]
            if rng.random() < 0.7:
                a = add(a, 1 if rng.random() < 0.5 else a)
            add(b, a)
            continue
        a = 2 * int(rng.integers(max(0, n - window), n)) + int(rng.integers(0, 2))
        if kind < again + fold:
            b = [0, 1, a, a ^ 1][int(rng.integers(0, 4))]
        else:
            b = 2 * int(rng.integers(max(0, n - window), n)) + int(rng.integers(0, 2))
        add(a, b)
    n = len(f0)
    pos = 2 * rng.integers(max(0, n - window), n, 40) + rng.integers(0, 2, 40)
    return nPIs, np.array(f0, np.uint32), np.array(f1, np.uint32), pos.astype(np.uint32)


SHAPES = [(1, 1, 4, 0.0, 0.0), (2, 60, 200, 0.3, 0.2), (6, 1500, 300, 0.1, 0.4), (40, 1500, 40, 0.02, 0.3),
          (300, 20000, 3000, 0.01, 0.3), (2000, 300_000, 4000, 0.01, 0.1)]


@pytest.mark.parametrize("shape", SHAPES, ids=["%dx%d" % s[:2] for s in SHAPES])
@pytest.mark.parametrize("schedule", [0, culs_amd.GLS_ST_LEVELS])
def test_strash_of_redundant_graphs(gpu_ctx, shape, schedule):
    print("whole strash:", shape, schedule)
    sys.stdout.flush()
    g = redundant(*shape, 9)
    a = gpu_ctx.from_arrays(*g).strash(schedule=schedule)
    print("final_strash", a.last_op()["final_strash"], "rounds", a.last_op()["strash_rounds"])
    want, depth = O.strash(*g)
    assert same(a.arrays(), want) and a.stats().levels == depth
    if schedule:
        assert a.last_op()["final_strash"] == 1
    # the levels it leaves, which a rewrite starts from, are the wave sweep's
    b = gpu_ctx.from_arrays(*g).strash(schedule=culs_amd.GLS_ST_WAVES)
    assert same(a.rewrite().arrays(), b.rewrite().arrays())


def test_batched_strash_of_redundant_graphs(gpu_ctx):
    print("whole strash of a batch")
    sys.stdout.flush()
    graphs = [redundant(*s, 20 + i) for i, s in enumerate(SHAPES[:5])]
    aigs = [gpu_ctx.from_arrays(*g) for g in graphs]
    gpu_ctx.batch_strash(aigs)
    for a, g in zip(aigs, graphs):
        want, depth = O.strash(*g)
        assert same(a.arrays(), want) and a.stats().levels == depth


def twice(nPIs, f0, f1, pos):
    """The ANDs of a graph twice over the same PIs, found equal level by level."""
    n, first = len(f0), nPIs + 1

    def copy(x):
        x = np.asarray(x, np.uint32)
        return np.where(x >> 1 >= first, x + 2 * (n - first), x).astype(np.uint32)

    return (nPIs, np.concatenate([f0, copy(f0[first:])]), np.concatenate([f1, copy(f1[first:])]),
            np.concatenate([pos, copy(pos)]))


# 2^18 objects and more than 128 rounds: on narrow levels the rounds go on (the
# waves are swept early then), on wide ones the wave sweep takes over
@pytest.mark.parametrize("pis,window,path", [(64, 300, 1), (1000, 3000, 2)], ids=["narrow", "wide"])
def test_strash_of_many_rounds(gpu_ctx, pis, window, path):
    print("whole strash, many rounds:", pis, window)
    sys.stdout.flush()
    g = twice(*gpu_ctx.gen_random(pis, 150_000, 50, window, 4).arrays())
    a = gpu_ctx.from_arrays(*g).strash()
    want, depth = O.strash(*g)
    print("depth", depth, "final_strash", a.last_op()["final_strash"], "rounds", a.last_op()["strash_rounds"])
    assert same(a.arrays(), want) and a.stats().levels == depth
    assert a.last_op()["final_strash"] == path
    b = gpu_ctx.from_arrays(*g).strash(schedule=culs_amd.GLS_ST_WAVES)
    assert same(a.rewrite().arrays(), b.rewrite().arrays())


@pytest.mark.parametrize("leaves", [1, 2047, 2048, 2049, 9000])
def test_dangling_cones(gpu_ctx, leaves):
    """A tree of ANDs that nothing refers to: its cascade's rounds are as wide as
    its levels, which fit a workgroup's queue up to 2048; beside it a live chain
    that has ANDs of a second dangling tree between its own."""
    print("dangling cones:", leaves)
    sys.stdout.flush()
    nPIs = 200
    rng = np.random.default_rng(leaves)
    f0, f1 = [0] * (nPIs + 1), [0] * (nPIs + 1)

    def add(a, b):
        f0.append(int(a))
        f1.append(int(b))
        return 2 * (len(f0) - 1)

    def lit():
        return 2 * int(rng.integers(1, nPIs + 1)) + int(rng.integers(0, 2))

    def tree(row):
        while len(row) > 1:
            row = [add(row[i], row[i + 1] ^ 1) if i + 1 < len(row) else row[i] for i in range(0, len(row), 2)]

    tree([add(lit(), lit()) for _ in range(leaves)])
    chain, second = add(lit(), lit()), []
    for _ in range(3000):
        second.append(add(chain ^ 1, lit()))
        chain = add(chain, lit())
    tree(second)
    g = nPIs, np.array(f0, np.uint32), np.array(f1, np.uint32), np.array([chain, chain ^ 1, 2], np.uint32)
    want, depth = O.strash(*g)
    for schedule in (0, culs_amd.GLS_ST_WAVES, culs_amd.GLS_ST_LEVELS):
        a = gpu_ctx.from_arrays(*g).strash(schedule=schedule)
        assert same(a.arrays(), want) and a.stats().levels == depth, schedule
