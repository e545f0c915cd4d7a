"""Settings where they have a part: the wave sweep's under a schedule that runs
it, the lines of rw's final strash and of the balance on both sides; and the
autotuner leaves alone what runs the same code under every candidate value."""
import sys

import numpy as np
import pytest

import culs_amd
import oracle_ffi as O

pytestmark = pytest.mark.gpu

DEFAULTS = {"cut_wide": 2048, "rw_sweep_width": 1024, "strash_table_factor": 4, "strash_wave_batch": 4,
            "balance_narrow_max": 4096}


def log(*a):
    print(*a)
    sys.stdout.flush()


def same(a, b):
    return all(np.array_equal(np.asarray(x), np.asarray(y)) for x, y in zip(a, b))


@pytest.fixture
def tuned(gpu_ctx):
    yield lambda **setting: gpu_ctx.set_tuning(-1, **setting)
    gpu_ctx.set_tuning(-1, **DEFAULTS)


@pytest.mark.parametrize("setting", [{"strash_table_factor": 8}, {"strash_wave_batch": 1}, {"strash_wave_batch": 64}],
                         ids=lambda d: "%s=%d" % next(iter(d.items())))
def test_wave_sweep(gpu_ctx, tuned, setting):
    log("wave sweep under", setting)
    for g in (gpu_ctx.gen_random(64, 20000, 32, 1000, 1).arrays(), gpu_ctx.gen_random(512, 60000, 100, 20000, 2).arrays()):
        tuned(**setting)
        a = gpu_ctx.from_arrays(*g).strash(schedule=culs_amd.GLS_ST_WAVES)
        want, depth = O.strash(*g)
        assert a.last_op()["final_strash"] == 0 and same(a.arrays(), want) and a.stats().levels == depth
        b = a.copy().rewrite(full_strash=True)
        assert b.last_op()["final_strash"] == 0 and same(b.arrays(), O.rw(*want)[0])


@pytest.mark.parametrize("width,route", [(1, 0), (1 << 30, 1)])
def test_final_strash_of_rw(gpu_ctx, tuned, width, route):
    log("rw_sweep_width", width)
    a = gpu_ctx.gen_random(64, 20000, 32, 1000, 1).strash()
    g = a.arrays()
    assert len(g[1]) > 8 * a.stats().levels
    tuned(rw_sweep_width=width)
    a.rewrite()
    assert a.last_op()["final_strash"] == route and same(a.arrays(), O.rw(*g)[0])


@pytest.mark.parametrize("narrow_max", [1, 1999, 2000, 2048])
def test_balance_line(gpu_ctx, tuned, narrow_max):
    """Levels of 2000 covers of two inputs, which fit the workgroup's LDS."""
    log("balance_narrow_max", narrow_max)
    rng = np.random.default_rng(1)
    nPIs, covers, layers = 50, 2000, 6
    f0, f1 = [np.zeros(nPIs + 1, np.int64)], [np.zeros(nPIs + 1, np.int64)]
    n, below = nPIs + 1, 2 * np.arange(1, nPIs + 1)
    for _ in range(layers):
        f0.append(rng.choice(below, covers) + 1)
        f1.append(rng.choice(below, covers) + 1)
        below = 2 * (n + np.arange(covers))
        n += covers
    f0, f1 = np.concatenate(f0), np.concatenate(f1)
    g = (nPIs, np.minimum(f0, f1).astype(np.uint32), np.maximum(f0, f1).astype(np.uint32), below.astype(np.uint32))
    tuned(balance_narrow_max=narrow_max)
    a = gpu_ctx.from_arrays(*g).balance(update_level=False)
    assert same(a.arrays(), O.balance(*g))


def test_autotune_leaves_what_has_no_part(gpu_ctx, tuned):
    a = gpu_ctx.gen_random(16, 2000, 8, 200, 3)
    a.simulate(words=1)
    assert a.copy().strash().last_op()["final_strash"] == 1
    objects = a.stats().nObjs
    tuned(strash_table_factor=8, strash_wave_batch=64)
    start = gpu_ctx.get_tuning(objects)
    for _ in range(5):
        best, best_ms, start_ms = gpu_ctx.autotune([a], culs_amd.GLS_TUNE_STRASH, reps=1)
        log("autotune strash", best, best_ms, start_ms)
        assert best == start and best_ms == start_ms


def test_autotune_tries_different_balances(gpu_ctx, tuned):
    """From 2048 on every narrow limit is the same."""
    a = gpu_ctx.gen_random(16, 2000, 8, 200, 3)
    a.simulate(words=1)
    for _ in range(5):
        tuned(balance_narrow_max=4096)
        best = gpu_ctx.autotune([a], culs_amd.GLS_TUNE_BALANCE, reps=1)[0]
        log("autotune balance", best)
        # (2048 only after a smaller one has been the fastest)
        assert best["balance_narrow_max"] in (256, 1024, 2048, 4096)
