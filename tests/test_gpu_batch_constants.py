"""Batched rw of members that refer to the constant: POs that are constant, ANDs
left dangling.  A cut whose table depends on fewer leaves than its cone has
reaches PIs and, through them, the constant, whose references are the member's
own and not the batch's.  Every member as if alone, against the oracle."""
import sys

import numpy as np
import pytest

import oracle_ffi as O

pytestmark = pytest.mark.gpu


def same(a, b):
    return all(np.array_equal(np.asarray(x), np.asarray(y)) for x, y in zip(a, b))


def member(rng, constants):
    """A strashed random AIG over few PIs, with constant POs besides its own."""
    nPIs, window = int(rng.integers(3, 9)), int(rng.choice([4, 12, 40]))
    f0, f1 = [0] * (nPIs + 1), [0] * (nPIs + 1)
    for _ in range(int(rng.integers(1, 60))):
        n = len(f0)
        a, b = 2 * rng.integers(max(0, n - window), n, 2) + rng.integers(0, 2, 2)
        f0.append(int(min(a, b)))
        f1.append(int(max(a, b)))
    n = len(f0)
    pos = np.concatenate([2 * rng.integers(max(0, n - 8), n, 3), rng.integers(0, 2, constants)]).astype(np.uint32)
    g = O.strash(nPIs, np.array(f0, np.uint32), np.array(f1, np.uint32), pos)[0]
    return g if same(O.strash(*g)[0], g) else member(rng, constants)


@pytest.mark.parametrize("zeros", [False, True])
@pytest.mark.parametrize("constants", [0, 1, 2, 5])
def test_batch_rewrite_with_constants(gpu_ctx, constants, zeros):
    print("batched rw, constants:", constants, zeros)
    sys.stdout.flush()
    rng = np.random.default_rng(constants)
    # the first half refers to the constant, the others do not
    graphs = [member(rng, constants if i < 200 else 0) for i in range(400)]
    aigs = [gpu_ctx.from_arrays(*g) for g in graphs]
    gpu_ctx.batch_strash(aigs)
    assert all(same(a.arrays(), g) for a, g in zip(aigs, graphs))
    gpu_ctx.batch_rewrite(aigs, use_zeros=zeros)
    wrong = [i for i, (a, g) in enumerate(zip(aigs, graphs)) if not same(a.arrays(), O.rw(*g, use_zeros=zeros)[0])]
    assert not wrong, wrong
