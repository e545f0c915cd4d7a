"""Selection of non-overlapping rewrites against the oracle where it takes many
rounds: redundant multipliers from a few candidates to thousands, so that one
workgroup takes over after the first round, later, or never."""
import sys

import numpy as np
import pytest

import oracle_ffi as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bits", [2, 3, 5, 8, 14, 22, 32, 48])
@pytest.mark.parametrize("redundant", [0.02, 0.3])
def test_selection_rounds(gpu_ctx, bits, redundant):
    a = gpu_ctx.gen_multiplier(bits, redundant, bits).strash()
    for zeros in (False, True):
        x = a.arrays()
        a.rewrite(use_zeros=zeros)
        print("selection: %d bits, %d rounds" % (bits, a.last_op()["rounds"]))
        sys.stdout.flush()
        want, stats = O.rw(*x, use_zeros=zeros)
        assert all(np.array_equal(np.asarray(p), np.asarray(q)) for p, q in zip(a.arrays(), want))
        assert a.last_op()["candidates"] == stats[0] and a.last_op()["selected"] == stats[1]
