"""Strash of graphs whose classes take a new least id in round after round, so
that every round brings as many new keys as there are ANDs: the table of keys
is emptied before it fills up; and of graphs that need more rounds than are worth
it.  Array for array against the oracle."""
import sys

import numpy as np
import pytest

import culs_amd
import oracle_ffi as O

pytestmark = pytest.mark.gpu


def falling(drops, fanouts):
    """Two equal chains of `drops` ANDs, found equal one AND per round.  For each
    of these an AND that equals x once it is: the least id of x's class falls in
    every round, and each of x's fanouts gets another key."""
    nPIs = 40 + (fanouts + 1) // 2
    f0, f1 = [0] * (nPIs + 1), [0] * (nPIs + 1)

    def add(a, b):
        f0.append(min(a, b))
        f1.append(max(a, b))
        return 2 * (len(f0) - 1)

    def pi(i):
        return 2 * (1 + i)

    chains = []
    for _ in range(2):
        cur, chain = pi(0), []
        for k in range(drops):
            cur = add(cur, pi(1 + k % 30) ^ (k // 30 & 1))
            chain.append(cur)
        chains.append(chain)
    u, v = pi(35), pi(36)
    # AND(p, not q) is constant once p and q are found equal
    copies = [add(add(u, add(p, q ^ 1) ^ 1), v) for p, q in reversed(list(zip(*chains)))]
    x = add(u, v)
    pos = [add(x, pi(40 + j // 2) ^ (j & 1)) for j in range(fanouts)] + copies
    return nPIs, np.array(f0, np.uint32), np.array(f1, np.uint32), np.array(pos, np.uint32)


@pytest.mark.parametrize("drops,fanouts", [(40, 2000), (30, 180_000)])
def test_keys_of_many_rounds(gpu_ctx, drops, fanouts):
    print("strash table:", drops, fanouts)
    sys.stdout.flush()
    g = falling(drops, fanouts)
    a = gpu_ctx.from_arrays(*g).strash(schedule=culs_amd.GLS_ST_LEVELS)
    op = a.last_op()
    print("final_strash", op["final_strash"], "rounds", op["strash_rounds"], "probes", op["hash_probes"])
    want, depth = O.strash(*g)
    assert all(np.array_equal(x, y) for x, y in zip(a.arrays(), want)) and a.stats().levels == depth
    assert op["final_strash"] == 1 and op["strash_rounds"] > drops
    # linear probing at seven eighths takes 32.5 probes for a new key on
    # average, and one more counts the least id; at most every AND per round
    assert op["hash_probes"] <= 34 * op["strash_rounds"] * (len(g[1]) - g[0] - 1)


def test_wide_graph_of_many_rounds(gpu_ctx):
    """At least 2^18 objects, the same logic twice on wide levels: after a few
    rounds the wave sweep is the faster way, and a part of the levels tells."""
    print("strash, wide levels, many rounds")
    sys.stdout.flush()
    nPIs, f0, f1, pos = gpu_ctx.gen_random(1000, 150_000, 50, 30_000, 4).arrays()
    up = 2 * (len(f0) - nPIs - 1)

    def copy(x):
        return np.where(x >> 1 > nPIs, x + up, x).astype(np.uint32)

    g = (nPIs, np.concatenate([f0, copy(f0[nPIs + 1:])]), np.concatenate([f1, copy(f1[nPIs + 1:])]),
         np.concatenate([pos, copy(pos)]))
    a = gpu_ctx.from_arrays(*g).strash()
    want, depth = O.strash(*g)
    assert all(np.array_equal(x, y) for x, y in zip(a.arrays(), want)) and a.stats().levels == depth
    assert a.last_op()["final_strash"] == 2
