"""The work that users of this library have it do, as measurable cases.

Each case is one command (or script of commands) on seeded synthetic AIGs
through the public Python API: the graph kinds are the library's generators,
the sizes are those of its tests (2,000 ANDs), of its benchmark (the 20,000-AND
random AIG, the 32-bit multiplier, the 10M-AND deep AIG, the mixed batch, the
`b; rw; rwz; b` jobs) and sizes between them.  A pass ends with the result's
arrays on the host, which is how a program gets a network back (`write`, gput),
in arrays that the program keeps; no pass gives back more objects than the
input had, so these are sized by the input, and what lies past the result's
objects stays zero.

Graphs are whole numbers throughout, so results are compared for equality and
`exact` has nothing to add.
"""
import ctypes
import math

import numpy as np

import culs_amd

CONVENTION = culs_amd.GLS_LIT_AIGER

_ctx = None
_server = None


def context():
    """The process's device context: a program opens one and keeps it."""
    global _ctx
    if _ctx is None:
        _ctx = culs_amd.Context(0)
    return _ctx


def server():
    """The process's rewrite server, kept for every request stream."""
    global _server
    if _server is None:
        _server = culs_amd.Server(0, hbm_budget=64 << 30, max_active=4096)
    return _server


def listed():
    return [
        # The smallest calls: a test-sized cone that an optimisation loop
        # rewrites in place, bound by launches and host round trips.
        {"name": "rw-2k", "op": "rw", "graph": "random", "ands": 2_000, "pis": 16, "pos": 8, "window": 200},
        # Load a network, `st; rw`, write it back: the ordinary script on an
        # ordinary (wide and shallow) AIG.
        {"name": "st-rw-20k", "op": "load_st_rw", "graph": "random", "ands": 20_000, "pis": 64, "pos": 32,
         "window": 1_000},
        # `st; rw; rwz` on arithmetic logic with redundancy: the multiplier.
        {"name": "mult32-st-rw-rwz", "op": "load_st_rw_rwz", "graph": "multiplier", "bits": 32, "redundant": 0.1},
        # A resynthesis script on a larger multiplier: balance between rewrites.
        {"name": "mult64-b-rw-rwz-b", "op": "b_rw_rwz_b", "graph": "multiplier", "bits": 64, "redundant": 0.1},
        # One pass of rw on a deep AIG with narrow levels, of odd size.
        {"name": "rw-deep-200k", "op": "rw", "graph": "geometric", "ands": 200_003, "pis": 1_024, "pos": 4_096,
         "window": 50_000, "p": 0.001},
        # Zero-gain rewriting of a large reconvergent AIG.
        {"name": "rwz-random-1m", "op": "rwz", "graph": "random", "ands": 1_000_000, "pis": 256, "pos": 2_500,
         "window": 5_000},
        # The headline: rw on the strashed 10M-AND deep AIG.
        {"name": "rw-deep-10m", "op": "rw", "graph": "geometric", "ands": 10_000_000, "pis": 1_024, "pos": 4_096,
         "window": 50_000, "p": 0.001},
        # Structural hashing of a raw 10M-AND AIG that is on the device.
        {"name": "st-deep-10m", "op": "st", "graph": "geometric", "ands": 10_000_000, "pis": 1_024, "pos": 4_096,
         "window": 50_000, "p": 0.001},
        # Balance of an AIG as large as the largest job of the serving mix.
        {"name": "b-random-2m", "op": "b", "graph": "random", "ands": 2_000_000, "pis": 256, "pos": 5_000,
         "window": 5_000},
        # Many independent AIGs of uneven size in one batched rw.
        {"name": "batch-rw-512", "op": "batch_rw", "graph": "mix", "count": 512, "least": 1_000, "most": 200_000},
        # A burst of jobs to the server, random AIGs and multipliers.
        {"name": "serve-32", "op": "serve", "graph": "jobs", "count": 32, "least": 1_000, "most": 2_000_000},
        # Simulation signatures of a rewritten network's outputs.
        {"name": "simulate-500k", "op": "simulate", "graph": "random", "ands": 500_000, "pis": 256, "pos": 1_250,
         "window": 1_000, "words": 64},
    ]


def _log_int(rng, least, most):
    return int(round(math.exp(rng.uniform(math.log(least), math.log(most)))))


def draw(rng):
    """One more case: an operation, a graph kind and sizes over the ranges
    that the listed cases span (log-uniform, so odd sizes are the rule)."""
    op = rng.choice(["rw", "rw", "rwz", "load_st_rw", "load_st_rw_rwz", "b_rw_rwz_b", "st", "b", "b_s", "batch_rw",
                     "serve", "simulate"])
    if op == "batch_rw":
        return {"op": op, "graph": "mix", "count": _log_int(rng, 4, 256), "least": _log_int(rng, 300, 3_000),
                "most": _log_int(rng, 10_000, 200_000)}
    if op == "serve":
        return {"op": op, "graph": "jobs", "count": _log_int(rng, 4, 32), "least": _log_int(rng, 300, 3_000),
                "most": _log_int(rng, 50_000, 1_000_000)}
    kind = rng.choice(["random", "geometric", "multiplier"])
    case = {"op": op, "graph": kind}
    if op == "simulate":
        case["words"] = rng.randint(1, 64)
    # the balance and the scripts on graphs of the serving mix's sizes, the
    # single passes up to a few million ANDs
    script = op.startswith("b")
    if kind == "multiplier":
        return {**case, "bits": rng.randint(8, 64 if script else 96), "redundant": round(rng.uniform(0.02, 0.3), 3)}
    ands = _log_int(rng, 1_000, 300_000 if script else 4_000_000 if op in ("rw", "st") else 1_000_000)
    if kind == "random":
        return {**case, "ands": ands, "pis": _log_int(rng, 16, 512), "pos": max(1, ands // 400),
                "window": _log_int(rng, 200, 5_000)}
    return {**case, "ands": ands, "pis": _log_int(rng, 32, 1_024), "pos": max(1, ands // 2_500),
            "window": _log_int(rng, 2_000, 50_000), "p": round(math.exp(rng.uniform(math.log(0.001), math.log(0.02))), 5)}


def mix_sizes(case):
    """AND counts of a batch or of a job list, evenly spread in the logarithm."""
    n = case["count"]
    span = math.log(case["most"] / case["least"])
    return [int(case["least"] * math.exp(span * (i + 0.5) / n)) for i in range(n)]


def job_kinds(case):
    """(kind, size) of every job: random AIGs and multipliers in turn; a
    multiplier's width stays within 8..64 bits."""
    sizes = mix_sizes(case)
    return [("random", n) if i % 2 else ("multiplier", 8 + (i * 56) // max(1, len(sizes) - 1))
            for i, n in enumerate(sizes)]


def _random(ctx, ands, seed):
    pis = max(16, ands // 200)
    return ctx.gen_random(pis, ands, max(1, pis // 2), 1_000, seed)


def _graph(ctx, case, seed):
    if case["graph"] == "multiplier":
        return ctx.gen_multiplier(case["bits"], case["redundant"], seed)
    if case["graph"] == "random":
        return ctx.gen_random(case["pis"], case["ands"], case["pos"], case["window"], seed)
    return ctx.gen_geometric(case["pis"], case["ands"], case["pos"], case["window"], case["p"], seed)


def _room(case):
    """(objects, POs) that every input of the case fits in, whatever its seed."""
    if case["graph"] in ("mix", "jobs"):
        shapes = [(n, "random") for n in mix_sizes(case)] if case["graph"] == "mix" else \
            [(n, kind) for kind, n in job_kinds(case)]
        rooms = [_mult_room(n, 0.05) if kind == "multiplier" else _random_room(n) for n, kind in shapes]
        return sum(r[0] for r in rooms), sum(r[1] for r in rooms)
    if case["graph"] == "multiplier":
        return _mult_room(case["bits"], case["redundant"])
    return 1 + case["pis"] + case["ands"], case["pos"]


def _mult_room(bits, redundant):
    return 1 + 2 * bits + int(10 * bits * bits * (1 + 2 * redundant)), 2 * bits


def _random_room(ands):
    pis = max(16, ands // 200)
    return 1 + pis + ands, max(1, pis // 2)


def prepare(case, seed):
    ctx, op = context(), case["op"]
    seed = 1 + int(seed) * 100_003
    objs, pos = _room(case)
    state = {"case": case, "f0": np.zeros(objs, np.uint32), "f1": np.zeros(objs, np.uint32),
             "pos": np.zeros(pos, np.uint32)}
    if op == "batch_rw":
        aigs = [_random(ctx, n, seed + i) for i, n in enumerate(mix_sizes(case))]
        ctx.batch_strash(aigs)
        return {**state, "aigs": aigs}
    if op == "serve":
        jobs = [(_random(ctx, n, seed + i) if kind == "random" else ctx.gen_multiplier(n, 0.05, seed + i)).arrays()
                for i, (kind, n) in enumerate(job_kinds(case))]
        return {**state, "jobs": jobs, "server": server()}
    aig = _graph(ctx, case, seed)
    if op.startswith("load"):
        return {**state, "arrays": aig.arrays()}
    if op in ("st", "simulate"):
        aig.simulate(words=1)       # puts the raw network on the device
        return {**state, "aig": aig}
    return {**state, "aig": aig.strash()}


def _at(array, k):
    return ctypes.c_void_p(array.ctypes.data + 4 * k)


def _collect(state, aigs):
    """The AIGs' arrays one after the other in the state's arrays, and how many
    objects they hold."""
    lib, f0, f1, pos = culs_amd.lib(), state["f0"], state["f1"], state["pos"]
    i = j = 0
    for a in aigs:
        s = a.stats()
        a.ctx.check(lib.gls_aig_to_arrays(a._h, _at(f0, i), _at(f1, i), _at(pos, j), CONVENTION), "gls_aig_to_arrays")
        i += s.nObjs
        j += s.nPOs
    return [i, f0.view(np.int32), f1.view(np.int32), pos.view(np.int32)]


def _serve(state):
    srv, lib, f0, f1, pos = state["server"], culs_amd.lib(), state["f0"], state["f1"], state["pos"]
    ids = [srv.submit(g, "b; rw; rwz; b") for g in state["jobs"]]
    i = j = 0
    for job in ids:
        info = srv.wait(job)
        if lib.gls_server_result(srv._h, job, _at(f0, i), _at(f1, i), _at(pos, j), CONVENTION) != 0:
            raise culs_amd.GlsError("gls_server_result failed")
        srv.release(job)
        i += 1 + info["nPIs"] + info["nAnds"]
        j += info["nPOs"]
    return [i, f0.view(np.int32), f1.view(np.int32), pos.view(np.int32)]


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "serve":
        return _serve(state)
    if op == "simulate":
        return state["aig"].simulate(words=case["words"], seed=7).view(np.int64)
    if op == "batch_rw":
        aigs = [a.copy() for a in state["aigs"]]
        context().batch_rewrite(aigs)
        return _collect(state, aigs)
    if op.startswith("load"):
        aig = context().from_arrays(*state["arrays"], CONVENTION).strash().rewrite()
        if op == "load_st_rw_rwz":
            aig.rewrite(use_zeros=True)
        return _collect(state, [aig])
    aig = state["aig"].copy()
    if op == "rw":
        aig.rewrite()
    elif op == "rwz":
        aig.rewrite(use_zeros=True)
    elif op == "st":
        aig.strash()
    elif op == "b":
        aig.balance()
    elif op == "b_s":
        aig.balance(shuffle=True)
    elif op == "b_rw_rwz_b":
        aig.balance().rewrite().rewrite(use_zeros=True).balance()
    else:
        raise ValueError(op)
    return _collect(state, [aig])


def _ands(case):
    if case["graph"] == "multiplier":
        # per cell a partial product and a full adder (two XORs, one majority)
        return int(9 * case["bits"] ** 2 * (1 + case["redundant"]))
    if case["graph"] == "mix":
        return sum(mix_sizes(case))
    if case["graph"] == "jobs":
        return sum(n if kind == "random" else 9 * n * n for kind, n in job_kinds(case))
    return case["ands"]


def work(case):
    """Two fanin literals of every AND read once and written once (whole
    numbers, no floating operations); for a simulation its AND operations on
    64-bit words instead of the second half."""
    ands = _ands(case)
    if case["op"] == "simulate":
        return {"bytes": 8 * ands, "flops": ands * case["words"]}
    return {"bytes": 16 * ands, "flops": 0}


def exact(case, seed):
    return None
