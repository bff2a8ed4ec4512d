"""What this framework is timed on: the calls that placement searches and serving studies make, through the public
entry points, from one small placement to the whole headline batch.

Every case has a ``kind`` (the entry point and what the program around it does) and its sizes:

  single      ``approximate_one_case_one_placement``: one placement, finish time and flag of every request
  one_case    ``approximate_one_case`` with its default (full) statistics: one serving case, percentiles per model
  scores      ``PlacementEvaluator.get_scores``: what a beam search asks for its candidates
  stats       ``PlacementEvaluator.get_stats``: what the evolutionary search and the greedy search without look-ahead ask
  successors  ``engine.evaluate_successors``: a greedy search that looks one step ahead
  replacing   ``PlacementEvaluator.get_stats`` on placements that replace one another during the workload
  seeds       ``engine.evaluate``: candidates on several arrival seeds in one call
  batch       ``engine.Batch``: a batch that stays on the device and is run and fetched

Models, arrivals and placements are drawn as the five benchmark configurations draw them
(``mms_amd.synthetic``): Gamma arrivals per model, power-law rates, evenly split pipelines; all from the seed.
"""
import math
from functools import partial

import numpy as np

from mms_amd import _lib, engine
from mms_amd.placement_policy import (ClusterEnv, ModelData, ModelPlacement, ModelPlacementWithReplacement,
                                      PlacementEvaluator)
from mms_amd.profiling import ParallelConfig, synthetic_profile
from mms_amd.simulator.controller import approximate_one_case, approximate_one_case_one_placement
from mms_amd.simulator.executable import Executable
from mms_amd.simulator.workload import Request, Workload
from mms_amd.synthetic import gamma_arrivals_fast, power_law_rates
from mms_amd.util import ServingCase

# Depth and operator-parallel degrees of a group, by the layout's name: "sr" selective replication (every device a
# group of its own), "pp4" equal four-stage pipelines, "mixed" groups of 1 to 8 devices as one pipeline each, "ops"
# groups of 2 to 16 devices split between operator and pipeline parallelism.
LAYOUTS = {"sr": ((1,), (1,)), "pp4": ((4,), (1,)), "mixed": ((1, 2, 4, 8), (1,)), "ops": ((2, 4, 8, 16), (1, 2, 4))}


def listed():
    return [
        # One placement on a minute of Poisson traffic (configuration 1): the smallest call there is, as a study that
        # plots single serving cases makes it.
        case("one placement, 1.2k requests", "single", "pp4", 8, 8, 1, 20.0, 60.0, 1.0, 0.0, 8, 8, slo=5.0),
        # The default statistics of one serving case on a training workload of the generator's minimum length
        # (30000 requests).
        case("one case, full statistics", "one_case", "mixed", 32, 16, 1, 60.0, 500.0, 4.0, 0.6, 4, 8, slo=5.0),
        # Candidates on four arrival seeds (configuration 2).
        case("64 candidates, 4 seeds", "seeds", "mixed", 32, 16, 64, 32.0, 300.0, 4.0, 0.0, 2, 6, seeds=4, slo=5.0),
        # A step of the greedy search with look-ahead: the current placement and every placement it can lead to, on
        # the training workload of the 32-model problem.
        case("greedy step, looking ahead", "successors", "sr", 32, 32, 700, 60.0, 1800.0, 4.0, 0.6, 1, 3, slo=5.0),
        # A step of the beam search over eight four-stage groups on the same workload.
        case("beam step, pipelines", "scores", "pp4", 32, 32, 600, 60.0, 1800.0, 4.0, 0.6, 3, 7, slo=5.0),
        # Every one-replica step from two placements of single-device groups (configuration 3).
        case("4096 replica steps", "scores", "sr", 64, 32, 4096, 200.0, 600.0, 2.0, 0.5, 3, 4, slo=8.0),
        # The population of the evolutionary search: 1024 children and the best so far, 64 models on 64 devices.
        case("population of 1025", "stats", "mixed", 64, 64, 1025, 120.0, 900.0, 4.0, 0.6, 2, 8, slo=5.0),
        # Placements that are replaced every 150 seconds, scored together.
        case("8 replacing placements", "replacing", "sr", 32, 16, 8, 60.0, 900.0, 4.0, 0.6, 2, 4, segments=6, slo=5.0),
        # The batching simulator behind an evaluator: a beam step of a study with dynamic batching.
        case("batching, 128 candidates", "scores", "mixed", 48, 24, 128, 60.0, 500.0, 4.0, 0.8, 4, 12, batching=True, slo=5.0),
        # The large batching set (configuration 5, a quarter of its candidates and of its time).
        case("batching, 2048 x 4 seeds", "batch", "mixed", 96, 48, 2048, 500.0, 300.0, 6.0, 0.8, 4, 12, seeds=4,
             batching=True, slo=5.0),
        # Per-model and per-group counts of a large bursty set (configuration 4's candidates on one of its seeds).
        case("4096 with counts, 1M requests", "batch", "ops", 128, 64, 4096, 1000.0, 1000.0, 8.0, 1.0, 8, 24, counts=True, slo=5.0),
        # The headline: configuration 4 whole, 16384 candidates on eight bursty streams of a million requests.
        case("16384 x 8 seeds, 1M requests", "batch", "ops", 128, 64, 16384, 1000.0, 1000.0, 8.0, 1.0, 8, 24, seeds=8, slo=5.0),
    ]


def case(name, kind, layout, models, devices, placements, rate, duration, cv, alpha, k_lo, k_hi, seeds=1, segments=1,
         batching=False, counts=False, slo=5.0):
    """A case: ``rate`` requests per second over all models (power law ``alpha``) for ``duration`` seconds at
    coefficient of variation ``cv``; a group hosts between ``k_lo`` and ``k_hi`` models; a request may take ``slo``
    times its model's latency on one device."""
    c = dict(kind=kind, layout=layout, models=models, devices=devices, placements=placements, rate=rate,
             duration=duration, cv=cv, alpha=alpha, k_lo=k_lo, k_hi=k_hi, seeds=seeds, segments=segments,
             batching=batching, counts=counts, slo=slo)
    return dict(c, name=name) if name else c


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["single", "one_case", "scores", "scores", "stats", "successors", "replacing", "seeds", "batch", "batch"])
    batching = rng.random() < 0.25 and kind not in ("successors", "replacing")
    # (most placements, fewest and most requests of a stream)
    most, fewest, requests = {"single": (1, 300, 120_000), "one_case": (1, 3_000, 120_000), "scores": (4096, 3_000, 120_000),
                              "stats": (2048, 3_000, 120_000), "successors": (2000, 3_000, 120_000),
                              "replacing": (48, 3_000, 120_000), "seeds": (512, 1_000, 30_000),
                              "batch": (16384, 10_000, 1_000_000)}[kind]
    placements = log(max(1, most // 500), most)
    total = log(fewest, requests)
    seeds = rng.randint(2, 6) if kind == "seeds" else rng.randint(1, 4) if kind == "batch" else 1
    if batching:
        placements, total = max(1, placements // 4), max(fewest, total // 4)
    if kind == "batch":     # the whole of it stays below what the headline batch holds
        total = min(total, int(3.2e10 / (placements * seeds)))
    devices = log(4, 64)
    models = log(4, 128)
    layout = rng.choice(["sr", "pp4", "mixed", "ops"] if devices >= 8 else ["sr", "mixed"])
    rate = float(round(models * rng.uniform(0.8, 4.0), 1))
    k_lo = rng.randint(1, max(1, models // 8))
    c = case("", kind, layout, models, devices, placements, rate, round(total / rate, 1), rng.choice([1.0, 2.0, 4.0, 6.0, 8.0]),
             round(rng.uniform(0.0, 1.0), 2), k_lo, min(models, k_lo + rng.randint(1, 8)), seeds=seeds,
             segments=rng.randint(2, 8) if kind == "replacing" else 1, batching=batching,
             counts=kind == "batch" and rng.random() < 0.5, slo=rng.choice([2.0, 5.0, 8.0]))
    return c


# ---- inputs ---------------------------------------------------------------------------------------------------------

def _profiles(c, rng):
    sizes, ops = LAYOUTS[c["layout"]]
    configs = sorted({ParallelConfig(1, o, s // o) for s in (1,) + sizes for o in ops if s % o == 0})
    latencies = rng.uniform(0.05, 0.4, c["models"])
    sizes_of_batches = (1, 2, 4, 8, 16) if c["batching"] else (1,)
    return latencies, [synthetic_profile("m%d" % m, float(latencies[m]), configs, batch_sizes=sizes_of_batches,
                                         batch_slope=0.15 if c["batching"] else 0.0, stage_comm=0.002 if len(ops) > 1 else 0.0)
                       for m in range(c["models"])]


def _stream(c, latencies, seed):
    """Arrivals, model ids and float32 SLOs of all models, merged as ``Workload.merge`` merges them: the first
    ``rate * duration`` requests, as bursts put more or fewer of them into the time itself."""
    rates = power_law_rates(c["models"], c["rate"], c["alpha"])
    count, duration = int(c["rate"] * c["duration"]), c["duration"]
    while True:
        duration *= 1.2
        per_model = [gamma_arrivals_fast(rates[m], c["cv"], 0, duration, (seed * 1009 + m) % (1 << 32)) for m in range(c["models"])]
        if sum(len(a) for a in per_model) >= count:
            break
    times = np.concatenate(per_model)
    ids = np.repeat(np.arange(c["models"], dtype=np.int32), [len(a) for a in per_model])
    order = np.argsort(times)[:count]
    return times[order], ids[order], (c["slo"] * latencies).astype(np.float32)[ids[order]]


def _placements(c, rng, n):
    """n placements of the case's layout: devices dealt to groups (the same groups whatever the seed, so that results
    of two seeds have one shape), every group hosting k_lo to k_hi models."""
    sizes, ops = LAYOUTS[c["layout"]]
    configs = {(s, o): ParallelConfig(1, o, s // o) for s in (1,) + sizes for o in ops if s % o == 0}
    lo, hi, models = c["k_lo"], c["k_hi"], c["models"]
    out, rows, at = [], [], 0
    deal = np.random.default_rng(c["devices"])
    for _ in range(n):
        cfgs, members, left = [], [], c["devices"]
        while left > 0:
            fitting = [s for s in sizes if s <= left] or [1]
            size = fitting[int(deal.random() * len(fitting))]
            left -= size
            op = [o for o in ops if size % o == 0]
            cfgs.append(configs[size, op[int(deal.random() * len(op))]])
            if at == len(rows):     # models of the next 4096 groups: the first k of a random order
                keys = rng.random((4096, models), dtype=np.float32)
                top = np.argpartition(keys, hi - 1, axis=1)[:, :hi] if hi < models else np.argsort(keys, axis=1)
                rows, at = top.tolist(), 0
            members.append(rows[at][:lo + int(rng.random() * (hi - lo + 1))])
            at += 1
        out.append(ModelPlacement(cfgs, members))
    return out


def _replica_steps(c, rng, n):
    """n placements, each one replica more than one of a few base placements (every step of a greedy or beam search)."""
    bases = _placements(dict(c, k_hi=max(c["k_lo"], c["k_hi"] - 1)), rng, max(1, -(-n // (c["devices"] * c["models"]))) + 1)
    out = []
    while len(out) < n:
        base = bases[len(out) % len(bases)]
        g, m = int(rng.integers(len(base.group_models))), int(rng.integers(c["models"]))
        if m not in base.group_models[g]:
            out.append(base.add_model(g, m).normalize())
        elif c["models"] == len(base.group_models[g]):
            out.append(base.normalize())
    return out


def _workload(times, ids, slos):
    names = ["m%d" % m for m in range(int(ids.max()) + 1 if len(ids) else 0)]
    return Workload(times, [Request(names[m], None, s, i, {}) for i, (m, s) in enumerate(zip(ids.tolist(), slos.tolist()))])


# ---- one pass -------------------------------------------------------------------------------------------------------

def prepare(case, seed):
    c = case
    rng = np.random.default_rng(seed)
    latencies, profiles = _profiles(c, rng)
    kind = c["kind"]
    names = ["m%d" % m for m in range(c["models"])]
    if kind in ("batch", "seeds"):
        # streams, latency table and candidates on the device or packed, as a program keeps them; with "seeds" the
        # candidates are new in every call
        eng = engine.Engine.default()
        streams = [_stream(c, latencies, seed * 16 + s) for s in range(c["seeds"])]
        loads = [engine.DeviceWorkload(eng, t, m, s, c["models"]) for t, m, s in streams]
        table = engine.LatencyTable(profiles, [1, 2, 4, 8] if c["batching"] else [1])
        flags = (_lib.BATCHING if c["batching"] else 0) | (_lib.WANT_MODEL_COUNTS | _lib.WANT_GROUP_COUNTS if c["counts"] else 0)
        sols = _placements(c, rng, c["placements"])
        if kind == "seeds":
            return partial(engine.evaluate, eng, loads, table, sols, flags)
        return _RunBatch(engine.Batch(eng, loads, table, engine.pack_placements(sols, table), flags), loads)

    times, ids, slos = _stream(c, latencies, seed)
    if kind == "single":
        sol = _placements(c, rng, 1)[0]
        return partial(approximate_one_case_one_placement, sol, names, profiles, ids, slos, times, enable_batching=c["batching"])
    if kind == "successors":
        # the base placement and the (group, model) steps from it, in the order a search lists them
        eng = engine.Engine.default()
        base = _placements(c, rng, 1)[0]
        steps = [(g, m) for g in range(len(base.group_models)) for m in range(c["models"]) if m not in base.group_models[g]]
        steps = steps[:c["placements"]] or [(0, 0)]
        load = engine.DeviceWorkload(eng, times, ids, slos, c["models"])
        return partial(engine.evaluate_successors, eng, [load], engine.LatencyTable(profiles, [1]), [base], [0] * len(steps),
                       [g for g, _ in steps], [m for _, m in steps], _lib.WANT_MODEL_COUNTS | _lib.WANT_GROUP_COUNTS)

    workload = _workload(times, ids, slos)
    if kind == "one_case":
        sol = _placements(c, rng, 1)[0]

        def register(controller):
            for name, profile in zip(names, profiles):
                controller.register_model.remote(name, partial(Executable, profile))
        return partial(_full_statistics, ServingCase(register, lambda start=0: workload, lambda controller: sol),
                       c["models"], c["batching"])

    rates = power_law_rates(c["models"], c["rate"], c["alpha"])
    datas = [ModelData(names[m], float(c["slo"] * latencies[m]), float(rates[m]), c["cv"], profiles[m]) for m in range(c["models"])]
    evaluator = PlacementEvaluator(datas, ClusterEnv(c["devices"], 13 << 30), workload, "fast_simulator", False,
                                   enable_batching=c["batching"])
    if kind == "scores":
        return partial(_scores, evaluator, _replica_steps(c, rng, c["placements"]))
    if kind == "replacing":
        cuts = [c["duration"] * k / c["segments"] for k in range(c["segments"])]
        sols = [ModelPlacementWithReplacement(cuts, _placements(c, rng, c["segments"])) for _ in range(c["placements"])]
    else:
        sols = [s.normalize() for s in _placements(c, rng, c["placements"])]
    return partial(_stats, evaluator, sols)


def run(state):
    return state()


class _RunBatch:
    def __init__(self, batch, loads):
        self.batch, self.loads = batch, loads

    def __call__(self):
        self.batch.run()
        self.batch.sync()
        return self.batch.fetch()


def _scores(evaluator, sols):
    return np.array(evaluator.get_scores(sols))


def _stats(evaluator, sols):
    stats = evaluator.get_stats(sols)
    return {"goodput": np.array([s[0] for s in stats]), "model_goodput": np.array([s[1] for s in stats]),
            "group_requests": np.concatenate([s[2] for s in stats]), "latency_mean": np.array([s[3].latency_mean for s in stats])}


def _full_statistics(serving_case, num_models, batching):
    stats, _ = approximate_one_case(serving_case, enable_batching=batching)
    fields = ("num_requests", "goodput", "throughput", "latency_mean", "latency_std", "latency_p90", "latency_p99")
    per_model = np.zeros((num_models, len(fields)))     # rows by model: one that got no request has none
    for r in stats.per_model_stats:
        per_model[int(r.name[1:])] = [getattr(r, k) for k in fields]
    return {"per_model": per_model, "group_requests": np.array(stats.group_num_requests),
            "overall": np.array([stats.goodput, stats.latency_mean, stats.request_rate])}


# ---- what a pass cannot do without ----------------------------------------------------------------------------------

def work(case):
    """Bytes: 16 of every request of every stream (arrival, model, SLO) once, the placements (a byte per replica and per
    group) once, the outputs once.  Operations: of every request on every placement that hosts its model the additions
    and maxima of the pipeline and the choice among the replicas, 2 * stages + replicas + 3."""
    c = case
    requests = c["rate"] * c["duration"]
    sizes, ops = LAYOUTS[c["layout"]]
    pairs = [(s, o) for s in sizes if s <= c["devices"] for o in ops if s % o == 0]
    stages = sum(s // o for s, o in pairs) / len(pairs)
    groups = c["devices"] / (sum(s for s, _ in pairs) / len(pairs))
    hosted = groups * (c["k_lo"] + c["k_hi"]) / 2        # replicas of a placement
    share = 1 - (1 - (c["k_lo"] + c["k_hi"]) / 2 / c["models"]) ** groups       # of the models that are hosted at all
    lanes = c["placements"] * c["seeds"]
    evals = requests * lanes
    per_eval = 2 * stages + max(1.0, hosted / max(1.0, share * c["models"])) + 3
    out = 12 * lanes
    if c["kind"] == "single":
        out += 9 * evals
    if c["kind"] in ("stats", "successors", "replacing", "one_case") or c["counts"]:
        out += lanes * 8 * (c["models"] + groups)
    return {"bytes": 16 * requests * c["seeds"] + c["placements"] * c["segments"] * (hosted + groups) + out,
            "flops": evals * share * per_eval}


def tolerance(case):
    """Decisions are exact: counts, flags and finish times may not differ.  Sums and means of up to a million doubles,
    and what is derived from them, may be added up in another order."""
    if case["kind"] == "single":
        return "exact"
    return {"rel": 1e-12, "max": 1e-11, "differ": 0.0}
