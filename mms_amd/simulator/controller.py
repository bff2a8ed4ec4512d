"""The approximate serving simulator, evaluated on the GPU.

Drop-in for the fast-simulator half of the reference's
``alpa_serve/simulator/controller.py``: ``DummyController`` (:282-305),
``approximate_one_case`` (:308-407) and
``approximate_one_case_one_placement`` (:410-503).  The request loops the
reference JIT-compiles with numba (:561-628, :631-798) run as HIP kernels
behind ``libmmsim``; nothing here computes a simulation on the CPU.

The event-driven simulator of the same reference file (``Controller``,
``GroupManager``, ``Client``, ``simulate_one_case``, :30-279) is host code in
``mms_amd.simulator.event_sim``; its names are re-exported here, where the
reference has them.
"""
from functools import partial
from typing import Callable

import numpy as np

from mms_amd import _lib, engine as _engine
from mms_amd.profiling import ProfilingResult
from mms_amd.simulator.workload import (DEFAULT_WARMUP, PerModelStatsResult,
                                        StatsResult, Workload)
from mms_amd.util import ServingCase, batchsize_config, eps
from mms_amd.simulator.event_sim import Client, Controller, GroupManager, simulate_one_case  # noqa: F401


def install_remote_methods(obj):
    """Give every public method a ``.remote`` alias of itself, so code written
    against Ray actor handles can drive a plain object
    (reference simulator/util.py:9-16)."""
    for key in dir(obj):
        value = getattr(obj, key)
        if callable(value) and not key.startswith("_"):
            wrapped = partial(value)
            wrapped.remote = wrapped
            setattr(obj, key, wrapped)


class DummyController:
    """Collects name -> ProfilingResult from ``register_model`` calls and
    ignores everything else (controller.py:282-305)."""

    def __init__(self):
        self.name2profiling = {}
        install_remote_methods(self)

    def register_model(self, name: str, model_def: Callable):
        assert isinstance(model_def, partial)
        for a in model_def.args:
            if isinstance(a, ProfilingResult):
                self.name2profiling[name] = a
                break

    def create_mesh_group_manager(self, *args, **kwargs):
        pass

    def create_replica(self, *args, **kwargs):
        pass

    def sync(self):
        pass


def _placement_to_replica_table(placement, num_models):
    """m_id2g_id of controller.py:418-422: groups hosting each model, ascending."""
    group_models = placement.group_models
    num_groups = len(placement.group_configs)
    m_id2g_id = np.full((num_models, max(num_groups, 1)), -1, dtype=np.int32)
    fill = [0] * num_models
    for g_id, m_ids in enumerate(group_models):
        for m_id in m_ids:
            m_id2g_id[m_id][fill[m_id]] = g_id
            fill[m_id] += 1
    return m_id2g_id


def approximate_one_case_one_placement(placement, model_names, prof_ress, model_ids, slos,
                                       arrivals, mixed=True, enable_batching=False):
    """Simulate one placement on one request stream; returns
    ``(start, finish, good, model_num_requests, model_num_good_requests,
    group_num_requests, group_num_good_requests)`` as controller.py:410-503.

    The stage-latency table follows :467-476 (and :451-461 with batching); the
    request loop runs on the GPU through the C ABI's single-placement calls.
    """
    eng = _engine.Engine.default()
    group_configs = placement.group_configs
    num_groups = len(group_configs)
    num_models = len(model_names)
    if num_groups == 0:
        raise ValueError("placement has no groups")   # np.max([]) in the reference (:465)
    arrivals = np.asarray(arrivals, dtype=np.float64)
    num_requests = len(arrivals)
    m_id2g_id = _placement_to_replica_table(placement, num_models)
    if not mixed:
        # one clock per group: largest and summed stage latency of every (model, group), with the
        # pipeline penalty, rounded to float32 on assignment (:433-443, :496-499)
        group_max_latency = np.empty((num_models, num_groups), dtype=np.float32)
        group_sum_latency = np.empty((num_models, num_groups), dtype=np.float32)
        for m_id in range(num_models):
            for g_id in range(num_groups):
                value = prof_ress[m_id].para_dict.get(group_configs[g_id], None)
                if value:
                    penalty = 0.009 * len(value.latency[1])
                    group_max_latency[m_id][g_id] = max(value.latency[1]) * (1 + penalty)
                    group_sum_latency[m_id][g_id] = sum(value.latency[1]) * (1 + penalty)
                else:
                    group_max_latency[m_id][g_id] = group_sum_latency[m_id][g_id] = np.inf
        finish = np.empty(num_requests, dtype=np.float64)
        good = np.empty(num_requests, dtype=bool)
        counts = _engine.simulate_requests(eng, finish, good, arrivals, model_ids, slos, m_id2g_id,
                                           group_max_latency, group_sum_latency, num_requests)
        return (arrivals, finish, good) + tuple(counts)
    num_stages = np.array([c.pp for c in group_configs], dtype=np.int32)
    max_num_stages = int(np.max(num_stages))
    batch_sizes = list(batchsize_config) if enable_batching else [1]

    table = _engine.LatencyTable(prof_ress, batch_sizes)
    cols = [table.config_id(c) for c in group_configs]
    lat, _ = table.arrays()                       # [M][C][Smax][NB]
    stage_latency = np.ascontiguousarray(lat[:, cols, :max_num_stages, :])

    start = arrivals
    finish = np.empty(num_requests, dtype=np.float64)
    good = np.empty(num_requests, dtype=bool)
    if enable_batching:
        g_id2m_id = np.full((num_groups, num_models), -1, dtype=np.int32)
        fill = [0] * num_groups
        for m_id, g_ids in enumerate(m_id2g_id):          # :424-430
            for g_id in g_ids:
                if g_id >= 0:
                    g_id2m_id[g_id][fill[g_id]] = m_id
                    fill[g_id] += 1
        counts = _engine.simulate_requests_mixed_batching(
            eng, finish, good, arrivals, model_ids, slos, m_id2g_id, g_id2m_id, num_stages,
            stage_latency, batch_sizes, num_requests)
    else:
        counts = _engine.simulate_requests_mixed(
            eng, finish, good, arrivals, model_ids, slos, m_id2g_id, num_stages,
            stage_latency[..., 0], num_requests)
    return (start, finish, good) + tuple(counts)


def replacement_cuts(placement, arrivals):
    """Index ranges of the segments of a ModelPlacementWithReplacement: a new segment starts at the
    first arrival strictly later than the next change time (controller.py:345-365)."""
    arrivals = np.asarray(arrivals)
    in_order = bool(np.all(arrivals[1:] >= arrivals[:-1]) and np.all(arrivals[:1] == arrivals[:1]))  # (and no NaN)
    cuts = [0]
    at = 0          # an arrival starts one segment at most
    for time in placement.start_times[1:]:
        if in_order:
            at += int(np.searchsorted(arrivals[at:], time, side="right"))
        else:
            later = np.flatnonzero(arrivals[at:] > time)
            at = at + int(later[0]) if len(later) else len(arrivals)
        if at >= len(arrivals):
            break
        cuts.append(at)
        at += 1
    cuts.append(len(arrivals))
    return list(zip(cuts[:-1], cuts[1:]))


# Device copies of arrival slices a caller-provided cache of simulate_replacements may hold.
SEGMENT_CACHE_ENTRIES = 64


def simulate_replacements(sols, model_names, prof_ress, model_ids, slos, arrivals, flags=0,
                          enable_batching=False, table=None, workload_cache=None):
    """All segments of all ``ModelPlacementWithReplacement`` in ``sols`` as lanes of ONE GPU launch
    (``mmsim_eval_pairs``): segment k of candidate n is its placement simulated from idle clocks on
    its slice of the arrivals, as the reference does one after another (controller.py:345-391).

    Returns one dict per candidate: ``n_good``, ``latency_sum`` and, with the count flags,
    ``model_num_requests`` / ``model_num_good`` / ``group_num_requests`` / ``group_num_good`` summed
    over its segments (:385-391; the group axis is as wide as the candidate's widest placement), and
    with ``WANT_PER_REQUEST`` ``finish`` / ``good`` concatenated (:381-383).

    ``workload_cache``: a dict that keeps the device copies of the arrival slices between calls (keyed by
    slice; the oldest are closed beyond ``SEGMENT_CACHE_ENTRIES``).  Without one the copies made for this call
    are closed before it returns.  A segment whose simulation failed (batching simulator: ``status != 0``)
    raises ``MmsimError``.
    """
    eng = _engine.Engine.default()
    arrivals = np.asarray(arrivals, dtype=np.float64)
    if table is None:
        table = _engine.LatencyTable(prof_ress, list(batchsize_config) if enable_batching else [1])
    if enable_batching:
        flags |= _lib.BATCHING
    cache = {} if workload_cache is None else workload_cache
    streams, stream_index, lanes, stream_of, owner = [], {}, [], [], []
    try:
        for n, sol in enumerate(sols):
            for seg, (lo, hi) in enumerate(replacement_cuts(sol, arrivals)):
                if (lo, hi) not in stream_index:
                    if (lo, hi) in cache:
                        cache[(lo, hi)] = cache.pop((lo, hi))      # most recently used last
                    else:
                        cache[(lo, hi)] = _engine.DeviceWorkload(eng, arrivals[lo:hi], model_ids[lo:hi],
                                                                 slos[lo:hi], len(model_names))
                    stream_index[(lo, hi)] = len(streams)
                    streams.append(cache[(lo, hi)])
                lanes.append(sol.placements[seg])
                stream_of.append(stream_index[(lo, hi)])
                owner.append((n, lo, hi))
        out = _engine.eval_pairs(eng, streams, table, _engine.pack_placements(lanes, table), stream_of, flags)
    finally:
        if workload_cache is None:
            for w in cache.values():
                w.close()
        else:                       # keep the slices used last, close the device copies of the others
            for key in list(cache)[:max(0, len(cache) - max(SEGMENT_CACHE_ENTRIES, len(stream_index)))]:
                if key not in stream_index:
                    cache.pop(key).close()
    results = [None] * len(sols)
    for n, sol in enumerate(sols):
        mine = [k for k, o in enumerate(owner) if o[0] == n]
        res = {"n_good": int(out["n_good"][mine].sum()), "latency_sum": float(np.sum(out["latency_sum"][mine]))}
        for key in ("model_num_requests", "model_num_good"):
            if key in out:
                res[key] = out[key][mine].sum(axis=0)
        gmax = max(len(p.group_configs) for p in sol.placements)
        for key in ("group_num_requests", "group_num_good"):
            if key in out:
                res[key] = out[key][mine][:, :gmax].sum(axis=0)
        if "finish" in out:
            res["finish"] = np.concatenate([out["finish"][k, :owner[k][2] - owner[k][1]] for k in mine])
            res["good"] = np.concatenate([out["good"][k, :owner[k][2] - owner[k][1]] for k in mine])
        results[n] = res
    return results


def approximate_one_case(case: ServingCase, seed: int = 0, warmup: int = DEFAULT_WARMUP,
                         debug: bool = False, fast_stats: bool = False,
                         enable_batching: bool = False, per_request_arrays: bool = False):
    """Score one serving case with the approximate simulator
    (controller.py:308-407).  ``seed`` and ``debug`` are accepted and unused,
    as in the reference; ``warmup`` only matters when ``fast_stats`` is off.

    With ``fast_stats`` off the statistics of a ``ModelPlacement`` are computed on the GPU
    (``device_compute_stats``) and finish / good are never copied to the host;
    ``per_request_arrays=True`` takes the host path instead (``Workload.compute_stats`` on the copied
    arrays), which also fills the per-request arrays of each ``PerModelStatsResult``."""
    from mms_amd.placement_policy.base_policy import (ModelPlacement,
                                                      ModelPlacementWithReplacement)

    register_models, generate_workload, place_models = case
    workload = generate_workload()

    if workload.enable_simulator_cache and workload.cached_data:
        model_ids, slos, model_names, prof_ress = workload.cached_data
        placement = place_models(None)
    else:
        controller = DummyController()
        register_models(controller)
        placement = place_models(controller)
        # model id == registration order (:331-334)
        model_names, prof_ress = zip(*controller.name2profiling.items())
        name2id = {name: i for i, name in enumerate(model_names)}
        model_ids, slos = _engine.request_arrays(workload.requests, name2id)
        if workload.enable_simulator_cache:
            workload.cached_data = (model_ids, slos, model_names, prof_ress)

    arrivals = workload.arrivals
    if isinstance(placement, ModelPlacement) and not fast_stats and not per_request_arrays:
        return device_compute_stats(workload, [placement], model_names, prof_ress, model_ids, slos, warmup,
                                    enable_batching=enable_batching)[0], placement
    if isinstance(placement, ModelPlacement):
        (start, finish, good, model_num_requests, model_num_good_requests,
         group_num_requests, group_num_good_requests) = approximate_one_case_one_placement(
             placement, model_names, prof_ress, model_ids, slos, arrivals,
             enable_batching=enable_batching)
    elif isinstance(placement, ModelPlacementWithReplacement):
        # every segment starts from idle clocks on its own slice of the arrivals (:345-391); all segments are
        # lanes of one launch
        counts = _lib.WANT_MODEL_COUNTS | _lib.WANT_GROUP_COUNTS
        res = simulate_replacements([placement], model_names, prof_ress, model_ids, slos, arrivals,
                                    counts if fast_stats else counts | _lib.WANT_PER_REQUEST,
                                    enable_batching=enable_batching)[0]
        model_num_requests, model_num_good_requests = res["model_num_requests"], res["model_num_good"]
        group_num_requests, group_num_good_requests = res["group_num_requests"], res["group_num_good"]
        if fast_stats:      # the fast statistics only need the sums (:393-403)
            return replacement_fast_stats(model_names, arrivals, res), placement
        start, finish, good = arrivals, res["finish"], res["good"]
    else:
        raise TypeError(f"unsupported placement type: {type(placement)}")

    if fast_stats:
        stats = fast_stats_result(model_names, start, finish, good, model_num_requests,
                                  model_num_good_requests, group_num_requests)
    else:
        stats = workload.compute_stats(start, finish, good, warmup)
        stats.group_num_requests = tuple(group_num_requests)
    return stats, placement


def warmup_skip(arrivals, warmup):
    """Requests that Workload.compute_stats trims at either end (workload.py:312-314); 0: none."""
    if len(arrivals) > 1:
        return max(int(warmup / (arrivals[-1] - arrivals[0]) * len(arrivals)), 0)
    return 0


def device_compute_stats(workload, sols, model_names, prof_ress, model_ids, slos, warmup,
                         enable_batching=False, table=None, device_workload=None):
    """``Workload.compute_stats`` (workload.py:308-354) for every placement in ``sols``, with the
    per-request outputs left on the GPU: one launch simulates all placements, a second one
    (``mmsim_batch_model_stats``) reduces finish / good to per-model counts, first and last
    accepted arrival, latency mean / deviation and the two percentiles inside the warm-up window.

    Returns one ``StatsResult`` per placement.  Counts, goodput, throughput, p90 and p99 equal the
    reference's; means and deviations are within 1e-12 relative (compensated sums on the device,
    pairwise sums in numpy).  The per-request arrays of ``PerModelStatsResult`` (``latency``,
    ``request_starts``, ``request_finishes``) are ``None``: they never leave the device.
    """
    eng = _engine.Engine.default()
    arrivals = np.asarray(workload.arrivals, dtype=np.float64)
    R = len(arrivals)
    if table is None:
        table = _engine.LatencyTable(prof_ress, list(batchsize_config) if enable_batching else [1])
    flags = _lib.WANT_GROUP_COUNTS | _lib.WANT_PER_REQUEST | (_lib.BATCHING if enable_batching else 0)
    own = device_workload is None
    dw = _engine.DeviceWorkload(eng, arrivals, model_ids, slos, len(model_names)) if own else device_workload
    packed = _engine.pack_placements(sols, table)
    skip = warmup_skip(arrivals, warmup)
    options = None
    try:
        # The statistics are taken from what the run leaves on the device, so a batching simulation that runs out
        # of idle-event slots (the reference's heap has no bound, the kernel's list is sized from the group count)
        # sends the whole batch round again with twice the slots.
        for attempt in range(6):
            batch = _engine.Batch(eng, [dw], table, packed, flags, options=options)
            try:
                batch.run()
                batch.sync()
                try:
                    out = batch.fetch(per_request=False)
                except _lib.MmsimError as err:
                    if err.code != _lib.E_OVERFLOW or attempt == 5:
                        raise
                    options = dict(getattr(eng, "_options", {}), batching_event_slots=2 * batch.info()["event_slots"])
                    continue
                ms = batch.model_stats([skip])
                break
            finally:
                batch.close()
    finally:
        if own:
            dw.close()

    lo, hi = (skip, R - skip) if skip > 0 else (0, R)
    ids = np.asarray(model_ids[lo:hi])
    n_window = len(ids)
    # models in the order of their first request inside the window, then (stable) by request count
    # (workload.py:321-327); a request of a model that was never registered (id -1) is listed under its name
    entries = {}
    placed, first_at = np.unique(ids[ids >= 0], return_index=True)
    first_at = np.nonzero(ids >= 0)[0][first_at] if len(placed) else first_at
    for m, at in zip(placed, first_at):
        entries[model_names[m]] = [int(at), 0, int(m)]
    for i in np.nonzero(ids < 0)[0]:
        name = workload.requests[lo + int(i)].model_name
        if name not in entries:
            entries[name] = [int(i), 0, -1]
        entries[name][1] += 1
    ordered = sorted(entries.items(), key=lambda kv: kv[1][0])
    interval = arrivals[hi - 1] - arrivals[lo]

    results = []
    for b, sol in enumerate(sols):
        st = {k: v[0, b] for k, v in ms.items()}
        rows = []
        for name, (_, count, m) in ordered:
            if m < 0:
                rows.append(PerModelStatsResult(name, count, np.float64(0), 0, np.float64(0), np.float64(0),
                                                0, 0, None, None, None))
                continue
            n_req, n_good = int(st["model_num_requests"][m]), int(st["model_num_good"][m])
            goodput = np.float64(n_good) / n_req
            throughput = n_good / (st["last_start"][m] - st["first_start"][m]) if n_good > 0 else 0
            rows.append(PerModelStatsResult(name, n_req, goodput, throughput, st["latency_mean"][m],
                                            st["latency_std"][m], st["latency_p90"][m], st["latency_p99"][m],
                                            None, None, None))
        rows.sort(key=lambda r: r.num_requests)     # stable
        total_good = int(st["model_num_good"].sum())
        stats = StatsResult(rows, tuple(out["group_num_requests"][0, b][:len(sol.group_configs)]),
                            np.float64(total_good) / n_window, np.sum(st["latency_sum"]) / n_window,
                            n_window, n_window / interval)
        results.append(stats)
    return results


def replacement_fast_stats(model_names, arrivals, res):
    """fast_stats_result from the sums over a candidate's segments: mean(good) = accepted / requests,
    mean(finish - start) = latency sum / requests (rejected requests contribute 0, :613-622)."""
    R = len(arrivals)
    interval = arrivals[-1] - arrivals[0]
    mreq, mgood = res["model_num_requests"], res["model_num_good"]
    per_model = [PerModelStatsResult(model_names[i], mreq[i], mgood[i] / (mreq[i] + eps), mreq[i] / interval,
                                     0, 0, 0, 0, [], [], []) for i in range(len(model_names))]
    return StatsResult(per_model, tuple(res["group_num_requests"]), np.float64(res["n_good"]) / R,
                       res["latency_sum"] / R, R, R / interval)


def fast_stats_result(model_names, start, finish, good, model_num_requests,
                      model_num_good_requests, group_num_requests):
    """The no-warmup statistics of controller.py:393-403."""
    interval = start[-1] - start[0]
    per_model = [PerModelStatsResult(
        model_names[i], model_num_requests[i],
        model_num_good_requests[i] / (model_num_requests[i] + eps),
        model_num_requests[i] / interval, 0, 0, 0, 0, [], [], [])
        for i in range(len(model_names))]
    return StatsResult(per_model, tuple(group_num_requests), np.mean(good),
                       np.mean(finish - start), len(start), len(start) / interval)
