"""Plans and new nodes with 4 to 64 candidates to a wavefront (the number doubles
with every doubling of the candidates above 8,192), against the oracle."""
import sys

import numpy as np
import pytest

import oracle_ffi as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ands", [300, 20_000, 120_000, 250_000, 600_000])
def test_rewrite_by_candidates(gpu_ctx, ands):
    a = gpu_ctx.gen_random(64, ands, max(1, ands // 400), 3_000, 8).strash()
    g = a.arrays()
    a.rewrite(use_zeros=True)
    print("plan lanes:", ands, "candidates", a.last_op()["candidates"])
    sys.stdout.flush()
    want, _ = O.rw(*g, use_zeros=True)
    assert all(np.array_equal(np.asarray(x), np.asarray(y)) for x, y in zip(a.arrays(), want))
