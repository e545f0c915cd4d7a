"""Balance at the sizes where the sweep that gives covers their levels changes
its way: chunks of 1024 covers, 15 chunks of levels in LDS (covers whose inputs
are further away), more than 6144 inputs in a chunk; with unreached covers, bit
for bit against the oracle, alone and as a member of a batch."""
import sys

import numpy as np
import pytest

import oracle_ffi as O

pytestmark = pytest.mark.gpu


def covers_at(distances, covers, k, seed, chain=0):
    """`covers` covers of k inputs, each with complemented earlier covers at one
    of the distances as inputs (PIs where there is none); `chain`: that many
    covers at the end have the one before as input.  Every third of the last
    covers drives a PO, so some covers are not reached."""
    rng = np.random.default_rng(seed)
    nPIs = 40
    f0, f1, tops = [0] * (nPIs + 1), [0] * (nPIs + 1), []
    for c in range(covers):
        lits = [2 * int(rng.integers(1, nPIs + 1)) + int(rng.integers(0, 2)) for _ in range(k)]
        for j in range(1, k):
            d = int(rng.choice(distances)) + int(rng.integers(0, 3))
            if c - d >= 0:
                lits[j] = tops[c - d] + 1
        if c and c >= covers - chain:
            lits[0] = tops[-1] + 1
        cur = lits[0]
        for x in lits[1:]:
            f0.append(cur)
            f1.append(x)
            cur = 2 * (len(f0) - 1)
        tops.append(cur)
    pos = np.array(tops[::-3][:max(1, covers // 30)], np.uint32)
    return nPIs, np.array(f0, np.uint32), np.array(f1, np.uint32), pos


CASES = {
    "one": ([1], 1, 2, 0), "chunk-1": ([1, 50], 1023, 3, 20), "chunk": ([1, 50], 1024, 3, 1024),
    "chunk+1": ([1, 1022], 1025, 3, 1025), "ring": ([1, 1023, 14335, 15359, 16383], 20_000, 3, 100),
    "far": ([15_360, 16_384, 20_000], 40_000, 2, 10), "inputs": ([1, 700, 3_000], 3_000, 9, 50),
}


def same(a, b):
    return all(np.array_equal(np.asarray(x), np.asarray(y)) for x, y in zip(a, b))


@pytest.mark.parametrize("name", CASES)
def test_cover_levels(gpu_ctx, name):
    print("cover levels:", name)
    sys.stdout.flush()
    distances, covers, k, chain = CASES[name]
    g = covers_at(distances, covers, k, 3, chain)
    a = gpu_ctx.from_arrays(*g)
    a.balance(update_level=False)
    assert same(a.arrays(), O.balance(*g))


def test_cover_levels_of_a_batch(gpu_ctx):
    print("cover levels of a batch")
    sys.stdout.flush()
    graphs = [covers_at(d, c, k, 5 + i, chain) for i, (d, c, k, chain) in enumerate(CASES.values())]
    # a member without an AND
    graphs.insert(2, (3, np.zeros(4, np.uint32), np.zeros(4, np.uint32), np.array([2, 1], np.uint32)))
    aigs = [gpu_ctx.from_arrays(*g) for g in graphs]
    gpu_ctx.batch_balance(aigs, update_level=False)
    for a, g in zip(aigs, graphs):
        assert same(a.arrays(), O.balance(*g))
