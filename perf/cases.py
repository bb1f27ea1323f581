"""Performance cases of the framework, through its public entry points.

A case is one of seven kinds of work that a program has the engine do:

- ``run``: a whole NSGA-III or RVEA run, restarted with ``reset()`` and run to
  its last generation, as a multi-start study does;
- ``batch``: ``BatchNSGA3`` advancing many uneven runs by some generations;
- ``serve``: a ``Server`` that admits requests while others run, steps until
  they have finished and hands out their results;
- ``select``: one NSGA-III environmental selection (``kernels.nsga3_select``);
- ``rank``: one constrained non-dominated sort (``kernels.nds_rank``);
- ``reproduce``: mating, SBX and polynomial mutation (``kernels.reproduce``);
- ``mlp``: the seeded-MLP objective (``kernels.eval_mlp``).

Sizes are those of the benchmark and of the quality protocol, and ragged ones
between them.  Whole runs use objectives whose arithmetic is pinned bit for
bit (quadratic centers, DTLZ), since one different rounding of an objective
moves every later generation; the MLP objective is measured as a call of its
own, against 64 bits.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cuda-moea_amd"))

import cuda_moea as cm  # noqa: E402
from cuda_moea import kernels as K  # noqa: E402

PROBLEMS = {"DTLZ1": cm.DTLZ1, "DTLZ2": cm.DTLZ2, "DTLZ4": cm.DTLZ4, "DTLZ7": cm.DTLZ7, "C2DTLZ2": cm.C2DTLZ2}


def listed():
    return [
        # The smallest run: 92 individuals, 91 directions, 12 variables, 200 generations.  Latency and launches.
        {"name": "run_nsga3_n92", "kind": "run", "algorithm": "NSGA3", "problem": "quadratic", "n": 92, "m": 3,
         "d": 12, "gens": 200, "partitions": 12, "copy": 0.0},
        # The quality protocol's run: 1024 individuals on DTLZ2 in 12 variables, a fifth of its 500 generations.
        {"name": "run_nsga3_n1024_dtlz2", "kind": "run", "algorithm": "NSGA3", "problem": "DTLZ2", "n": 1024, "m": 3,
         "d": 12, "gens": 100, "partitions": 0, "copy": 0.5},
        # The headline run: 32768 individuals, 1024 variables, 20 generations.
        {"name": "run_nsga3_n32768_d1024", "kind": "run", "algorithm": "NSGA3", "problem": "quadratic", "n": 32768,
         "m": 3, "d": 1024, "gens": 20, "partitions": 0, "copy": 0.0},
        # RVEA at the benchmark's population and objective count, adaptive directions, on DTLZ2.
        {"name": "run_rvea_n16384_m5", "kind": "run", "algorithm": "RVEA", "problem": "DTLZ2", "n": 16384, "m": 5,
         "d": 2048, "gens": 10, "partitions": 0, "copy": 0.0},
        # 256 uneven runs (N 64 to 4096, M 3, 5 or 8, D 10 to 1000) advanced together by 50 generations.
        {"name": "batch_256", "kind": "batch", "count": 256, "gens": 50, "n_high": 4096, "d_high": 1000, "mixseed": 2024},
        # A served burst: 16 requests (N 64 to 8192, M 3 to 10, D 10 to 4096), half of them arriving mid-way.
        {"name": "serve_16", "kind": "serve", "count": 16, "gens": 40, "n_high": 8192, "d_high": 4096, "mixseed": 777},
        # The standalone selection of the benchmark: 65536 merged rows on a thick positive sphere shell, M = 3.
        {"name": "select_n32768_m3", "kind": "select", "n": 32768, "m": 3, "d": 2, "infeasible": 0.0, "grid": 0},
        # A many-objective selection of ragged size with infeasible rows.
        {"name": "select_n8190_m10", "kind": "select", "n": 8190, "m": 10, "d": 777, "infeasible": 0.1, "grid": 0},
        # A full ranking (every front) of an odd number of rows, with constraints and tied objective values.
        {"name": "rank_n20001_m5", "kind": "rank", "n": 20001, "m": 5, "infeasible": 0.2, "grid": 64, "half": False},
        # The dimension-bound reproduction of the RVEA benchmark.
        {"name": "reproduce_n16384_d131072", "kind": "reproduce", "n": 16384, "d": 131072, "copy": 0.0, "pm": 1.0},
        # The dimension-bound objective of the RVEA benchmark: an MLP D -> 256 -> 5.
        {"name": "mlp_n16384_d131072", "kind": "mlp", "n": 16384, "d": 131072, "hidden": 256, "m": 5},
        # The same objective at a served request's size, ragged.
        {"name": "mlp_n2046_d1333", "kind": "mlp", "n": 2046, "d": 1333, "hidden": 256, "m": 8},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _even(v):
    return v + (v & 1)


def draw(rng):
    kind = rng.choice(["run", "run", "batch", "serve", "select", "rank", "reproduce", "mlp"])
    if kind == "run":
        if rng.random() < 0.3:
            n, d = _log(rng, 64, 16384), _log(rng, 12, 2048)
            return {"kind": kind, "algorithm": "RVEA", "problem": rng.choice(["DTLZ1", "DTLZ2", "quadratic"]), "n": n,
                    "m": rng.choice([3, 5]), "d": d, "gens": 50 if n < 2048 else 10, "partitions": 0, "copy": 0.0}
        n, d = _even(_log(rng, 64, 32768)), _log(rng, 12, 1024)
        return {"kind": kind, "algorithm": "NSGA3",
                "problem": rng.choice(["quadratic", "DTLZ1", "DTLZ2", "DTLZ7", "C2DTLZ2"]), "n": n,
                "m": rng.choice([3, 3, 5, 8]), "d": d, "gens": 100 if n < 2048 else 10, "partitions": 0,
                "copy": rng.choice([0.0, 0.5])}
    if kind == "batch":
        return {"kind": kind, "count": _log(rng, 8, 256), "gens": 20, "n_high": _log(rng, 512, 4096),
                "d_high": _log(rng, 64, 1000), "mixseed": rng.randrange(1 << 20)}
    if kind == "serve":
        return {"kind": kind, "count": rng.randint(4, 16), "gens": 20, "n_high": _log(rng, 1024, 8192),
                "d_high": _log(rng, 64, 4096), "mixseed": rng.randrange(1 << 20)}
    if kind == "select":
        return {"kind": kind, "n": _even(_log(rng, 46, 32768)), "m": rng.choice([2, 3, 4, 5, 8, 10]),
                "d": _log(rng, 2, 512), "infeasible": rng.choice([0.0, 0.0, 0.1, 0.5]), "grid": rng.choice([0, 0, 32])}
    if kind == "rank":
        return {"kind": kind, "n": _log(rng, 100, 65536), "m": rng.choice([2, 3, 5, 8, 10]),
                "infeasible": rng.choice([0.0, 0.2]), "grid": rng.choice([0, 64]), "half": rng.random() < 0.5}
    if kind == "reproduce":
        n = _log(rng, 64, 16384)
        return {"kind": kind, "n": n, "d": _log(rng, 10, 131072), "copy": rng.choice([0.0, 0.5]),
                "pm": rng.choice([1.0, 1.0, 0.0])}
    return {"kind": kind, "n": _log(rng, 64, 16384), "d": _log(rng, 10, 131072), "hidden": rng.choice([128, 256]),
            "m": rng.choice([3, 5, 8, 10])}


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _problem(name, d, m, seed):
    return cm.QuadraticCenters(d, m, seed=seed) if name == "quadratic" else PROBLEMS[name](dimension=d, objectives=m)


def _mix(case, ms):
    """The uneven runs of a batch or a server: N and D log-uniform, M from ``ms``."""
    rng = np.random.default_rng(case["mixseed"])
    specs = []
    for _ in range(case["count"]):
        n = int(round(math.exp(rng.uniform(math.log(64), math.log(case["n_high"])))))
        m = int(rng.choice(ms))
        d = int(round(math.exp(rng.uniform(math.log(10), math.log(case["d_high"])))))
        specs.append((n + (n & 1), m, d))
    return specs


def _points(n, m, seed, infeasible, grid):
    """Objective rows s*u (u uniform on the positive part of the unit sphere, s in [1, 2]): many fronts.  ``grid``:
    values rounded to that many steps, so that rows tie.  cv: zero, or uniform for the infeasible part."""
    g = _gen(seed)
    u = torch.randn(n, m, generator=g, device="cuda").abs_()
    u /= u.norm(dim=1, keepdim=True)
    f = u * (1.0 + torch.rand(n, 1, generator=g, device="cuda"))
    if grid:
        f = torch.round(f * grid) / grid
    cv = torch.rand(n, generator=g, device="cuda")
    cv = torch.where(torch.rand(n, generator=g, device="cuda") < infeasible, cv, torch.zeros_like(cv))
    return f.t().contiguous(), cv


def prepare(case, seed):
    kind = case["kind"]
    if kind == "run":
        directions = {}
        if case["partitions"]:
            directions = {"reference_directions": cm.DasDennisDirections(partitions=case["partitions"])}
        alg = cm.Algorithm(case["algorithm"], population_size=case["n"], max_generations=case["gens"],
                           problem=_problem(case["problem"], case["d"], case["m"], seed), seed=seed,
                           crossover=cm.SBX(variable_copy_probability=case["copy"]), print_progress=False, **directions)
        alg.initialize()
        return {"kind": kind, "alg": alg}
    if kind == "batch":
        partitions = {3: 12, 5: 6, 8: 3}
        runs = [cm.NSGA3(population_size=n, max_generations=1_000_000, problem=cm.QuadraticCenters(d, m, seed=seed + i),
                         seed=seed + i, reference_directions=cm.DasDennisDirections(partitions=partitions[m]),
                         print_progress=False) for i, (n, m, d) in enumerate(_mix(case, [3, 5, 8]))]
        batch = cm.BatchNSGA3(runs)
        batch.initialize()
        return {"kind": kind, "batch": batch, "count": len(runs), "gens": case["gens"]}
    if kind == "serve":
        runs = [cm.NSGA3(population_size=n, max_generations=case["gens"] // (1 + i % 2),
                         problem=cm.QuadraticCenters(d, m, seed=seed + i), seed=seed + i, print_progress=False)
                for i, (n, m, d) in enumerate(_mix(case, [3, 5, 8, 10]))]
        for r in runs:
            r.problem.centers = r.problem.centers.cuda()      # payloads are resident before their requests arrive
        server = cm.Server(16 << 30, max_instances=32, max_rows=2 * 8192 * 32)
        return {"kind": kind, "server": server, "runs": runs, "late": case["gens"] // 4}
    if kind == "select":
        n, m, d = case["n"], case["m"], case["d"]
        f, cv = _points(2 * n, m, seed, case["infeasible"], case["grid"])
        x = torch.rand(2 * n, d, generator=_gen(seed + 1), device="cuda")
        half = [K.Population(x[s].contiguous(), f[:, s].contiguous(), cv[s].contiguous())
                for s in (slice(0, n), slice(n, 2 * n))]
        return {"kind": kind, "parents": half[0], "offspring": half[1], "seed": seed,
                "directions": torch.from_numpy(K.das_dennis(n, m)).cuda(),
                "ideal": f[:, :n].min(dim=1).values.contiguous()}
    if kind == "rank":
        f, cv = _points(case["n"], case["m"], seed, case["infeasible"], case["grid"])
        return {"kind": kind, "f": f, "cv": cv, "stop": case["n"] // 2 if case["half"] else None}
    if kind == "reproduce":
        n, d = case["n"], case["d"]
        x = torch.rand(n, d, generator=_gen(seed), device="cuda")
        bounds = torch.tensor([0.0, 1.0], device="cuda").repeat(d)
        rank = torch.randint(0, 24, (n,), generator=_gen(seed + 1), device="cuda", dtype=torch.int32)
        return {"kind": kind, "x": x, "bounds": bounds, "rank": rank, "cv": torch.zeros(n, device="cuda"),
                "copy": case["copy"], "pm": case["pm"], "seed": seed}
    x, w1, w2 = _mlp_inputs(case, seed)
    return {"kind": kind, "x": x, "w1": w1, "w2": w2}


def _mlp_inputs(case, seed):
    n, d, hidden, m = case["n"], case["d"], case["hidden"], case["m"]
    g = _gen(seed)
    x = torch.rand(n, d, generator=g, device="cuda")
    w1 = torch.randn(hidden, d, generator=g, device="cuda") / math.sqrt(d)
    w2 = torch.randn(m, hidden, generator=g, device="cuda") / math.sqrt(hidden)
    return x, w1, w2


def _flat(results):
    """The results of many runs as four tensors: variables, objectives, constraints, fronts."""
    return {"x": torch.cat([r.variables.reshape(-1) for r in results]),
            "f": torch.cat([r.objectives.reshape(-1) for r in results]),
            "cv": torch.cat([r.constraints.reshape(-1) for r in results]),
            "fronts": torch.cat([r.auxiliary_indices.reshape(-1) for r in results])}


def run(state):
    kind = state["kind"]
    if kind == "run":
        alg = state["alg"]
        alg.reset()
        r = alg.run(copy=False)
        if alg.kind == "NSGA3":
            return {"x": r.variables, "f": r.objectives, "cv": r.constraints, "fronts": r.auxiliary_indices}
        # rows past the active count hold NaN variables and sentinel objectives; the indices are those of front zero
        live = torch.arange(r.constraints.numel(), device=r.constraints.device) < r.active_count
        zero = torch.zeros((), device=r.constraints.device)
        front = torch.zeros_like(live)
        front[r.auxiliary_indices.long()] = True
        return {"x": torch.where(live[:, None], r.variables, zero), "f": torch.where(live[:, None], r.objectives, zero),
                "cv": torch.where(live, r.constraints, zero), "front": front, "active": int(r.active_count),
                "directions": alg.directions}
    if kind == "batch":
        batch = state["batch"]
        batch.step(state["gens"])
        return _flat([batch.result(i, copy=False) for i in range(state["count"])])
    if kind == "serve":
        server, runs = state["server"], state["runs"]
        first, late = runs[: len(runs) // 2], runs[len(runs) // 2:]
        slots = {server.admit(r): i for i, r in enumerate(first)}
        results, steps = [None] * len(runs), 0
        while slots:
            for slot in server.step():
                results[slots.pop(slot)] = server.result(slot)
                server.release(slot)
            steps += 1
            if steps == state["late"]:
                slots.update({server.admit(r): len(first) + i for i, r in enumerate(late)})
        return _flat(results)
    if kind == "select":
        ideal = state["ideal"].clone()                        # the selection updates it in place
        nxt, fronts, stats = K.nsga3_select(state["parents"], state["offspring"], state["directions"], ideal,
                                            seed=state["seed"], generation=1)
        return {"x": nxt.x, "f": nxt.f, "cv": nxt.cv, "fronts": fronts, "ideal": ideal, "counts": stats[:3]}
    if kind == "rank":
        fronts, last = K.nds_rank(state["f"], state["cv"], state["stop"])
        return {"fronts": fronts, "last": last}
    if kind == "reproduce":
        off, parents = K.reproduce(state["x"], state["bounds"], rank=state["rank"], cv=state["cv"],
                                   sbx=(30.0, 1.0, state["copy"]), pm=(20.0, state["pm"]), seed=state["seed"], generation=3)
        return {"x": off, "parents": parents}
    f, cv = K.eval_mlp(state["x"], state["w1"], state["w2"])
    return {"f": f, "cv": cv}


def _generation_work(n, m, d):
    """One generation of one run: parents read and offspring written by reproduction, survivors read and written by the
    selection; the objective's arithmetic (about 3 operations a variable and objective)."""
    return 16.0 * n * d, 3.0 * n * d * m


def work(case):
    kind = case["kind"]
    if kind == "run":
        b, f = _generation_work(case["n"], case["m"], case["d"])
        return {"bytes": case["gens"] * b, "flops": case["gens"] * f}
    if kind in ("batch", "serve"):
        each = [_generation_work(n, m, d) for n, m, d in _mix(case, [3, 5, 8] if kind == "batch" else [3, 5, 8, 10])]
        gens = [case["gens"] // (1 + i % 2) if kind == "serve" else case["gens"] for i in range(len(each))]
        return {"bytes": sum(g * b for g, (b, _) in zip(gens, each)), "flops": sum(g * f for g, (_, f) in zip(gens, each))}
    if kind == "select":
        n, m, d = case["n"], case["m"], case["d"]
        return {"bytes": 8.0 * n * d + 4.0 * (2 * n) * (m + 1) + 4.0 * n * (m + 2), "flops": 2.0 * n * m * m}
    if kind == "rank":
        n, m = case["n"], case["m"]
        return {"bytes": 4.0 * n * (m + 2), "flops": n * m * math.log2(n)}
    if kind == "reproduce":
        n, d = case["n"], case["d"]
        return {"bytes": 8.0 * n * d + 12.0 * n, "flops": 40.0 * n * d}
    n, d, h, m = case["n"], case["d"], case["hidden"], case["m"]
    return {"bytes": 4.0 * (n * d + h * d + h * m + n * (m + 1)), "flops": 2.0 * n * h * (d + m) + 3.0 * n * d}


def exact(case, seed):
    """The MLP objective in 64 bits.  The other kinds choose rows or draw them: their results are whole numbers and
    copied rows, or follow the engine's own generator, and have no other value to stand against."""
    if case["kind"] != "mlp":
        return None
    x, w1, w2 = _mlp_inputs(case, seed)
    w1, w2 = w1.double(), w2.double()
    rows = max(1, (1 << 28) // case["d"])
    f = []
    for i in range(0, case["n"], rows):
        xd = x[i:i + rows].double()
        f.append((torch.tanh(xd @ w1.t()) @ w2.t()).square().t() + 0.01 * (xd - 0.5).square().sum(dim=1))
    return {"f": torch.cat(f, dim=1), "cv": torch.zeros(case["n"], dtype=torch.float64, device="cuda")}
