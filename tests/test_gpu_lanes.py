"""The plain simulator with lanes at their own pace (sim_lanes.hip) against the CPU oracle, bit for bit, at the sizes where it can
go wrong: streams that end inside a block of 8192 requests or a segment, runs cut by a model, an SLO, a block or a request of no
model, arrivals out of order, models with none, one to four, five to eight and more replicas, depths that are powers of two and others,
infinite latencies and odd SLOs, items that take turns, placements with a stream of their own."""
from types import SimpleNamespace

import numpy as np
import pytest

from mms_amd import _lib, engine as E
from mms_amd.placement_policy.base_policy import ModelPlacement
from mms_amd.profiling import ParallelConfig
from oracle import oracle_c
from helpers import assert_batch_matches, oracle_batch
from test_gpu_window import _problem

pytestmark = pytest.mark.gpu

OWN = dict(skip_ahead=2, window_lanes=-1)


def _bursts(seed, R, M, load, odd_slos=True, ends=0.12):
    """Runs of 1 to some 30 requests of a model, its SLO mostly the same over a run."""
    rng = np.random.default_rng(seed)
    n = R + 1
    lengths = rng.geometric(ends, n)
    ids = np.repeat(rng.integers(-1, M, n), lengths)[:R].astype(np.int32)
    slos = np.repeat(rng.uniform(0.1, 0.9, n), lengths)[:R].astype(np.float32)
    if odd_slos:
        other = rng.random(R) < 0.03
        slos[other] = rng.choice(np.array([np.inf, np.nan, 0.25], dtype=np.float32), int(other.sum()))
    gaps = rng.exponential(0.02 / load, R) * (rng.random(R) > 0.3)
    return SimpleNamespace(tstamps=np.cumsum(gaps), model_ids=ids, slos=slos)


def _check(eng, streams, profiles, sols, M, options, expect="sim_lanes_kernel<"):
    table = E.LatencyTable(profiles, [1])
    packed = E.pack_placements(sols, table)
    dws = [E.DeviceWorkload(eng, s.tstamps, s.model_ids, s.slos, M) for s in streams]
    batch = E.Batch(eng, dws, table, packed, 0, options=options)
    assert batch.kernel_name().startswith(expect), batch.kernel_name()
    for _ in range(2):                                     # a second run starts from scratch again
        batch.run()
        batch.sync()
    out = batch.fetch()
    batch.close()
    for k, st in enumerate(streams):
        assert_batch_matches(out, oracle_batch(st, table, packed), k, packed[0], where=f"{options} stream {k}")
    for dw in dws:
        dw.close()


@pytest.mark.parametrize("depths,groups,hosts", [((1, 2, 4), 5, 4), ((1, 3, 4), 9, 5), ((1, 2, 4, 8, 16), 7, 4), ((1, 2, 16), 14, 5),
                                                 ((2, 5, 11), 12, 5), ((8, 32), 6, 4), ((7, 20), 6, 5)])
@pytest.mark.parametrize("options", [{}, dict(segment_requests=192, sched_groups=1, waves_per_cu=2)])
def test_lanes_at_their_own_pace(depths, groups, hosts, options):
    eng = E.Engine.default()
    M = 5 if groups > 6 else 9
    streams = [_bursts(k, R, M, 1.0 + k) for k, R in enumerate((0, 1, 63, 65, 8191, 8193, 17000))]
    for B in (1, 64, 131):
        profiles, sols = _problem(B + sum(depths), depths, True, M, groups, B, hosts)
        _check(eng, streams, profiles, sols, M, dict(OWN, **options))


def test_where_the_number_of_replicas_changes_the_path():
    """The first four replicas of a run are always there, the second four fetched where a model has them, and those beyond eight read in
    the step: 1 to 21 replicas of the model most asked for, beside models with one, two and none."""
    eng = E.Engine.default()
    rng = np.random.default_rng(3)
    profiles, _ = _problem(5, (1, 2, 4), True, 5, 1, 1, 1)
    pcs = [ParallelConfig(1, 1, d) for d in (1, 2, 4)]
    sols = []
    for n in (1, 2, 3, 4, 5, 7, 8, 9, 12, 16, 21):
        hosts = [set() for _ in range(22)]
        for m, k in ((0, n), (1, 1), (2, 2), (3, max(1, n - 4))):      # (model 4: nowhere)
            for g in rng.permutation(22)[:k]:
                hosts[g].add(m)
        for copies in range(3):
            sols.append(ModelPlacement([pcs[int(rng.integers(3))] for _ in hosts], [sorted(int(m) for m in h) for h in hosts]))
    streams = [_bursts(20 + k, R, 5, load) for k, (R, load) in enumerate(((3000, 3.0), (3000, 12.0), (3000, 60.0)))]
    _check(eng, streams, profiles, sols, 5, OWN)


def test_arrivals_out_of_order_and_runs_of_one_model():
    """The latest arrival of a run, not its last one, decides whether the rest of it is passed over; one model all along makes runs as
    long as a block; requests of no model alone make none."""
    eng = E.Engine.default()
    M = 6
    profiles, sols = _problem(11, (1, 2, 4), True, M, 6, 70, 3)
    mixed = _bursts(1, 5000, M, 8.0)
    rng = np.random.default_rng(2)
    shuffled = SimpleNamespace(tstamps=mixed.tstamps + rng.choice([0.0, 3.0], 5000) * (rng.random(5000) < 0.2), model_ids=mixed.model_ids, slos=mixed.slos)
    one = _bursts(3, 17000, M, 4.0, odd_slos=False)
    one.model_ids[:] = 2
    one.slos[:] = 0.4
    nobody = _bursts(4, 4200, M, 4.0)
    nobody.model_ids[:] = -1
    _check(eng, [shuffled, one, nobody], profiles, sols, M, OWN)


def test_a_stream_for_every_placement():
    eng = E.Engine.default()
    M = 7
    profiles, sols = _problem(21, (1, 2, 4, 8), True, M, 6, 200, 3)
    streams = [_bursts(40 + k, R, M, 6.0) for k, R in enumerate((9000, 8192, 0, 700))]
    table = E.LatencyTable(profiles, [1])
    packed = E.pack_placements(sols, table)
    dws = [E.DeviceWorkload(eng, s.tstamps, s.model_ids, s.slos, M) for s in streams]
    of = np.arange(200, dtype=np.int32) * 7 % 4
    with eng.options(**OWN):
        out = E.eval_pairs(eng, dws, table, packed, of)
    for k, st in enumerate(streams):
        ref = oracle_batch(st, table, packed)
        rows = np.flatnonzero(of == k)
        assert np.array_equal(out["n_good"][rows], ref["n_good"][rows])
        assert np.array_equal(out["latency_sum"][rows], ref["latency_sum"][rows])


@pytest.mark.parametrize("depths,load,expect", [((2, 4), 300.0, "sim_lanes_kernel<4, true>"), ((2, 4), 0.002, "sim_mixed_kernel<4,"),
                                                ((1,), 300.0, "sim_mixed_kernel<1,")])
def test_load_decides(depths, load, expect):
    eng = E.Engine.default()
    M = 20
    profiles, sols = _problem(31, depths, True, M, 4, 70, 2)
    _check(eng, [_bursts(50, 8200, M, load)], profiles, sols, M, dict(window_lanes=-1), expect)


@pytest.mark.parametrize("change,expect", [(0.0, "sim_lanes_kernel<4, true>"), (0.02, "sim_lanes_kernel<4, true>"), (0.4, "sim_mixed_kernel<4,"),
                                           (1.0, "sim_mixed_kernel<4,")])
def test_runs_of_one_slo_decide(change, expect):
    """A run ends where the SLO changes: bursts of a model whose requests have SLOs of their own are runs of one request each."""
    eng = E.Engine.default()
    M = 20
    profiles, sols = _problem(31, (2, 4), True, M, 4, 70, 2)
    st = _bursts(50, 8200, M, 300.0, odd_slos=False)
    new = np.random.default_rng(4).random(8200) < change
    st.slos[new] = np.linspace(0.2, 0.9, int(new.sum()), dtype=np.float32)
    _check(eng, [st], profiles, sols, M, dict(window_lanes=-1), expect)


@pytest.mark.parametrize("models,hosts,load,ends,expect", [(20, 2, 300.0, 0.12, "sim_lanes_kernel<4, true>"), (3, 3, 3000.0, 0.12, "sim_mixed_kernel<4,"),
                                                         (20, 0, 300.0, 0.12, "sim_mixed_kernel<4,"), (20, 2, 300.0, 0.04, "sim_mixed_kernel<4,")])
def test_replicas_and_bursts_decide(models, hosts, load, ends, expect):
    """Requests with many replicas, with none, and bursts of more than twenty requests on shallow groups keep the loop over runs, however
    large the load."""
    eng = E.Engine.default()
    profiles, sols = _problem(31, (2, 4), True, models, 12 if hosts == 3 else 4, 70, hosts)
    if hosts == 3:
        sols = [ModelPlacement(s.group_configs, [[0, 1, 2]] * len(s.group_models)) for s in sols]
    _check(eng, [_bursts(50, 8200, models, load, odd_slos=False, ends=ends)], profiles, sols, models, dict(window_lanes=-1), expect)


@pytest.mark.parametrize("options,expect", [(dict(request_loop=1), "sim_mixed_kernel<4, true, true, true, 0, true>"),
                                            (dict(request_loop=0), "sim_mixed_kernel<4, true, true, true, 0, false>"),
                                            (dict(request_loop=1, skip_ahead=2), "sim_lanes_kernel<4, true>"),
                                            (dict(request_loop=0, skip_ahead=2), "sim_mixed_kernel<4, true, true, true, 0, false>")])
def test_a_loop_that_is_asked_for_is_taken(options, expect):
    eng = E.Engine.default()
    profiles, sols = _problem(31, (2, 4), True, 20, 4, 70, 2)
    _check(eng, [_bursts(50, 8200, 20, 300.0)], profiles, sols, 20, dict(window_lanes=-1, **options), expect)


@pytest.mark.parametrize("what", ["items", "segments", "runs"])
def test_what_the_schedule_or_the_list_of_runs_cannot_hold_takes_the_loop_it_had(what):
    """Two in three requests repeat model and SLO, four in five do not: the loop without lanes at their own pace is the chunked one,
    which takes any number of (tile, stream) pairs, ignores the segments, and needs no list of runs (with 2^32 of them, refused
    after they were counted)."""
    eng = E.Engine.default()
    M = 20
    profiles, sols = _problem(31, (2, 4), True, M, 4, 70, 2)
    R, copies, options = {"items": (4100, 140, dict(sched_groups=1)),
                          "segments": (60010 * 64, 1, dict(sched_groups=1, waves_per_cu=1, segment_requests=64)),
                          "runs": (1 << 24, 257, dict(skip_ahead=2))}[what]
    st = _bursts(50, R, M, 300.0, odd_slos=False, ends=0.28)
    if what == "runs":      # every request a run of its own
        st.model_ids = (np.arange(R) % M).astype(np.int32)
    table = E.LatencyTable(profiles, [1])
    packed = E.pack_placements(sols, table)
    dw = E.DeviceWorkload(eng, st.tstamps, st.model_ids, st.slos, M)
    chunked = "sim_mixed_kernel<4, true, true, true, 0, false>"
    if what != "runs":      # (the streams alone are for lanes at their own pace)
        batch = E.Batch(eng, [dw], table, packed, 0, options=dict(window_lanes=-1))
        assert batch.kernel_name() == "sim_lanes_kernel<4, true>"
        batch.close()
    batch = E.Batch(eng, [dw] * copies, table, packed, 0, options=dict(window_lanes=-1, **options))
    assert batch.kernel_name() == chunked, batch.kernel_name()
    if what == "items":
        batch.run()
        batch.sync()
        out = batch.fetch()
        ref = oracle_batch(st, table, packed)
        for k in range(copies):
            assert_batch_matches(out, ref, k, packed[0], where=f"stream {k}")
    batch.close()
    dw.close()


def test_reported_bytes_are_those_that_the_kernel_reads():
    eng = E.Engine.default()
    M, R = 20, 20000
    profiles, sols = _problem(31, (2, 4), True, M, 4, 70, 2)
    table = E.LatencyTable(profiles, [1])
    st = _bursts(50, R, M, 300.0, odd_slos=False)
    dw = E.DeviceWorkload(eng, st.tstamps, st.model_ids, st.slos, M)
    batch = E.Batch(eng, [dw], table, E.pack_placements(sols, table), 0, options=OWN)
    starts = np.ones(R, bool)       # of the runs: a change of model or SLO, or of the block of 8192 requests
    starts[1:] = (st.model_ids[1:] != st.model_ids[:-1]) | (st.slos[1:] != st.slos[:-1]) | (np.arange(1, R) % 8192 == 0)
    runs = int((starts & (st.model_ids >= 0)).sum())
    info = batch.info()
    assert info["stream_bytes"] == 32 * (runs + 1) + 8 * R + 4 * (3 + 1) + 8      # runs (a spare one), arrivals, first run of a block, first block
    assert info["table_bytes"] == 2 * M * 2 * 64 * 8 + 8 * M * (len(table.arrays()[1]) + 1)      # entries, latencies of the configurations
    batch.close()
    dw.close()


@pytest.mark.parametrize("segment,segments", [(0, 3), (12288, 3), (8192, 6), (8256, 3), (4096, 11)])
@pytest.mark.parametrize("waves", [1, 2])
def test_items_that_take_turns_go_on_where_they_were(segment, segments, waves):
    """Segments of several blocks, the default one among them: a parked item goes on at the block that its segment starts with, its
    clocks and sums as they were.  Segments are whole numbers of blocks of 8192 requests, or one block if they are shorter."""
    eng = E.Engine.default()
    M = 6
    profiles, sols = _problem(41, (1, 2, 4, 8), True, M, 7, 131, 3)
    streams = [_bursts(60 + k, R, M, 3.0 + 3 * k) for k, R in enumerate((40961, 33001, 8191))]
    options = dict(OWN, sched_groups=1, waves_per_cu=waves, segment_requests=segment)
    table = E.LatencyTable(profiles, [1])
    dws = [E.DeviceWorkload(eng, s.tstamps, s.model_ids, s.slos, M) for s in streams]
    batch = E.Batch(eng, dws, table, E.pack_placements(sols, table), 0, options=options)
    info = batch.info()
    assert (info["segments"], info["workgroups"]) == (segments, 1), info
    batch.close()
    for dw in dws:
        dw.close()
    _check(eng, streams, profiles, sols, M, options)
