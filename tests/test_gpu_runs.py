"""Simulations cut into runs that are simulated at the same time (sim_window.hip) against the CPU oracle, bit for bit: streams
with pauses, in which neighbouring runs come to agree, streams that overload the groups all along, where none do and the first
run goes through the whole stream, and streams of both, where runs are given up and taken up again; streams that end inside a
span, at its edge and before it; all outputs."""
import ctypes as C
from contextlib import contextmanager
from types import SimpleNamespace

import numpy as np
import pytest

from mms_amd import _lib, engine as E
from mms_amd.placement_policy import ModelPlacement
from mms_amd.profiling import ParallelConfig
from helpers import assert_batch_matches, oracle_batch
from test_gpu_window import COUNTS, _problem, _stream

pytestmark = pytest.mark.gpu


def _with_pauses(seed, R, M, load, every, pause=4.0, quiet_until=1.0):
    """Pauses once in ``every`` requests, in the first ``quiet_until`` of the stream."""
    st = _stream(seed, R, M, load)
    rng = np.random.default_rng(seed + 1)
    gaps = np.diff(st.tstamps, prepend=0.0)
    gaps[(rng.random(R) < 1.0 / every) & (np.arange(R) < quiet_until * R)] += pause
    st.tstamps = np.cumsum(gaps)
    st.slos[np.isinf(st.slos) & (rng.random(R) < 0.97)] = 0.7      # (few: a clock that never comes down again never agrees)
    return st


def _busy_between(seed, R, M, load, first, end):
    """Pauses in which the groups catch up, but for the requests [first, end), which come ``load`` times as fast."""
    st = _with_pauses(seed, R, M, 0.6, 10 ** 9)
    rng = np.random.default_rng(seed + 2)
    gaps = np.diff(st.tstamps, prepend=0.0)
    busy = (np.arange(R) >= first) & (np.arange(R) < end)
    gaps[busy] *= 0.6 / load
    gaps[(rng.random(R) < 1.0 / 150) & ~busy] += 4.0
    st.tstamps = np.cumsum(gaps)
    st.slos = np.where(np.isfinite(st.slos), st.slos, np.float32(0.5))        # (a clock that an infinite one drove up stays up)
    return st


@pytest.mark.parametrize("depths,uniform,groups,hosts", [((1,), True, 6, 7), ((1, 2, 4), True, 6, 8), ((1, 3, 4), False, 9, 7)])
def test_runs_taken_up_again_meet_others(depths, uniform, groups, hosts):
    """Requests that overload several groups of every model for longer than a run may go on behind its span, twice, and pauses before,
    between and behind: runs are given up and taken up again, and those meet the runs that started in the pauses."""
    eng = E.Engine.default()
    M, span = 9, 512
    streams = [_busy_between(31 + k, 300 * 64 + 17, M, 3.0, 60 * 64, 170 * 64) for k in range(2)] + [_with_pauses(40, 200 * 64, M, 0.6, 100)]
    streams.append(_busy_between(33, 400 * 64, M, 3.0, 40 * 64, 130 * 64))
    late = _busy_between(34, 400 * 64, M, 3.0, 200 * 64, 290 * 64)
    gaps = np.diff(streams[3].tstamps, prepend=0.0)
    gaps[180 * 64:] = np.diff(late.tstamps, prepend=0.0)[180 * 64:]
    streams[3].tstamps = np.cumsum(gaps)
    dws = [E.DeviceWorkload(eng, s.tstamps, s.model_ids, s.slos, M) for s in streams]
    for B, flags in ((24, COUNTS), (9, COUNTS | _lib.WANT_PER_REQUEST), (40, 0)):
        profiles, sols = _problem(B + sum(depths), depths, uniform, M, groups, B, hosts)
        table = E.LatencyTable(profiles, [1])
        packed = E.pack_placements(sols, table)
        batch = E.Batch(eng, dws, table, packed, flags, options=dict(window_lanes=64, segment_requests=span))
        assert batch.kernel_name().count(",") == 6            # (the last one: cut into runs)
        outs = []
        for _ in range(3):
            batch.run()
            batch.sync()
            assert batch.info()["runs_met_again"] > 0
            outs.append(batch.fetch())
        batch.close()
        for k, st in enumerate(streams):
            ref = oracle_batch(st, table, packed, want_per_request=bool(flags & _lib.WANT_PER_REQUEST))
            for out in outs:
                if flags & _lib.WANT_PER_REQUEST:
                    R = len(st.tstamps)
                    assert np.array_equal(out["good"][k][:, :R], ref["good"]) and np.array_equal(out["finish"][k][:, :R], ref["finish"])
                assert_batch_matches(out, ref, k, packed[0], where=f"B={B}, stream {k}")
    for dw in dws:
        dw.close()


@pytest.mark.parametrize("depths,uniform,groups,hosts,M", [((1,), True, 6, 4, 9), ((1,), True, 40, 5, 5), ((1, 2, 4), True, 5, 4, 9),
                                                           ((1, 3, 4), False, 9, 5, 5), ((1, 2, 4, 8, 16), True, 7, 4, 9), ((8, 32), True, 6, 4, 9)])
@pytest.mark.parametrize("span", [512, 1024])
def test_runs_of_one_simulation(depths, uniform, groups, hosts, M, span):
    eng = E.Engine.default()
    streams = [_with_pauses(1, 7 * span + 333, M, 0.6, 150), _with_pauses(2, 8 * span, M, 4.0, 10 ** 9), _with_pauses(3, 7 * span + 1, M, 2.0, 200, quiet_until=0.6),
               _with_pauses(4, 3 * span, M, 1.0, 100), _with_pauses(5, 1, M, 1.0, 100), _with_pauses(6, 0, M, 1.0, 100)]
    dws = [E.DeviceWorkload(eng, s.tstamps, s.model_ids, s.slos, M) for s in streams]
    for B, flags in ((1, COUNTS | _lib.WANT_PER_REQUEST), (5, COUNTS), (40, 0)):
        profiles, sols = _problem(B + sum(depths), depths, uniform, M, groups, B, hosts)
        table = E.LatencyTable(profiles, [1])
        packed = E.pack_placements(sols, table)
        batch = E.Batch(eng, dws, table, packed, flags, options=dict(window_lanes=64, segment_requests=span))
        assert batch.kernel_name().count(",") == 6            # (the last one: cut into runs)
        for _ in range(3):                                 # further runs start from scratch again
            batch.run()
            batch.sync()
        out = batch.fetch()
        batch.close()
        for k, st in enumerate(streams):
            ref = oracle_batch(st, table, packed, want_per_request=bool(flags & _lib.WANT_PER_REQUEST))
            if flags & _lib.WANT_PER_REQUEST:
                R = len(st.tstamps)
                assert np.array_equal(out["good"][k][:, :R], ref["good"]) and np.array_equal(out["finish"][k][:, :R], ref["finish"])
            assert_batch_matches(out, ref, k, packed[0], where=f"B={B}, stream {k}")
    for dw in dws:
        dw.close()


def test_where_simulations_are_cut_by_themselves():
    """Few simulations of long streams, plain and paired; a latency sum that doubles many times, with half-way roundings."""
    eng = E.Engine.default()
    profiles, sols = _problem(3, (1, 2, 4), True, 9, 6, 12, 4)
    table = E.LatencyTable(profiles, [1])
    packed = E.pack_placements(sols, table)
    streams = [_with_pauses(11, 40000, 9, 0.8, 120), _with_pauses(12, 21000, 9, 0.8, 10 ** 9)]
    dws = [E.DeviceWorkload(eng, s.tstamps, s.model_ids, s.slos, 9) for s in streams]
    refs = [oracle_batch(s, table, packed) for s in streams]
    for flags in (0, COUNTS):
        batch = E.Batch(eng, dws, table, packed, flags)
        assert batch.kernel_name().count(",") == 6            # (the last one: cut into runs)
        batch.run()
        batch.sync()
        out = batch.fetch()
        batch.close()
        for k in range(2):
            assert_batch_matches(out, refs[k], k, packed[0], where=f"flags {flags}, stream {k}")
    of = np.arange(len(sols)) % 2
    got = E.eval_pairs(eng, dws, table, packed, of, COUNTS)
    for key in ("n_good", "latency_sum", "model_num_good", "group_num_requests", "group_num_good"):
        assert np.array_equal(got[key], np.where((of == 0).reshape((-1,) + (1,) * (refs[0][key].ndim - 1)), refs[0][key], refs[1][key])), key
    for dw in dws:
        dw.close()


@pytest.mark.parametrize("depths,uniform,groups,hosts,M", [((1,), True, 6, 4, 9), ((1, 2, 4), True, 9, 4, 9), ((1, 3, 5), False, 12, 6, 70), ((2, 8), True, 5, 9, 140)])
@pytest.mark.parametrize("span", [512, 1024])
def test_runs_of_the_batching_simulator(depths, uniform, groups, hosts, M, span):
    """Queues, idle events and models that no group lists as well.  Latencies are added up in another order than the oracle's: of n
    of them, none negative, both sums are within n * 2^-53 of the exact one (8525 requests: 9.5e-13)."""
    eng = E.Engine.default()
    streams = [_with_pauses(1, 7 * span + 333, M, 0.6, 150), _with_pauses(2, 8 * span, M, 4.0, 10 ** 9), _with_pauses(3, 7 * span + 1, M, 2.0, 200, quiet_until=0.6),
               _with_pauses(4, 3 * span, M, 1.0, 100), _with_pauses(5, 1, M, 1.0, 100), _with_pauses(6, 0, M, 1.0, 100)]
    for s in streams:
        s.slos = np.where(np.isfinite(s.slos), s.slos, np.float32(0.4))       # (an infinite one lets a clock become infinite: not supported)
    dws = [E.DeviceWorkload(eng, s.tstamps, s.model_ids, s.slos, M) for s in streams]
    sizes = [1, 2, 4, 8]
    for B, flags in ((1, COUNTS), (40, 0)):
        profiles, sols = _problem(B + sum(depths), depths, uniform, M, groups, B, hosts)
        for p in profiles:
            for d in p.para_dict.values():
                for b in sizes[1:]:
                    d.latency[b] = [x * (1 + 0.15 * (b - 1)) for x in d.latency[1]]
        table = E.LatencyTable(profiles, sizes)
        packed = E.pack_placements(sols, table)
        batch = E.Batch(eng, dws, table, packed, flags | _lib.BATCHING, options=dict(segment_requests=span))
        assert batch.kernel_name().startswith("sim_batching_solo_kernel<") and batch.kernel_name().count(",") == 4    # (the last one: cut into runs)
        outs = []
        for _ in range(3):
            batch.run()
            batch.sync()
            outs.append(batch.fetch())
        batch.close()
        for out in outs:
            assert not out["status"].any()
            for k, st in enumerate(streams):
                ref = oracle_batch(st, table, packed, batching=True)
                assert np.array_equal(out["n_good"][k], ref["n_good"]), (B, k)
                for key in ("model_num_good", "group_num_requests", "group_num_good") if flags else ():
                    assert np.array_equal(out[key][k], ref[key]), (B, k, key)
                assert np.array_equal(out["latency_sum"][k], outs[0]["latency_sum"][k]), (B, k)   # wherever the runs met
                assert np.allclose(out["latency_sum"][k], ref["latency_sum"], rtol=1e-12, atol=0), (B, k)
    for dw in dws:
        dw.close()


def test_clocks_that_no_request_can_tell_apart():
    """Groups that nobody asks for during a span (their clocks stay as they were, or at zero), in the same order and not, and an
    arrival that is earlier than the one before it, which takes the shortcut away."""
    eng = E.Engine.default()
    M, span, R = 8, 512, 6 * 512
    for uneven in (False, True):
        rng = np.random.default_rng(5)
        profiles, _ = _problem(5, (1, 2), True, M, 1, 1, 1)
        pcs = sorted({pc for p in profiles for pc in p.para_dict}, key=lambda c: c.pp)
        sols = [_problem(60 + k, (1, 2), True, M, 9, 1, 3)[1][0] for k in range(24)]
        # a phase for the first half of the models, one for the second, and so on; pauses within
        st = _with_pauses(21, R, M, 0.5, 40, pause=2.0)
        phase = np.arange(R) // 700 % 2
        st.model_ids = (rng.integers(0, M // 2, R) + phase * (M // 2)).astype(np.int32)
        st.slos = np.where(np.isfinite(st.slos), st.slos, np.float32(0.5))
        if uneven:
            st.tstamps[2000:] -= 3.0
        table = E.LatencyTable(profiles, [1])
        packed = E.pack_placements(sols, table)
        dw = E.DeviceWorkload(eng, st.tstamps, st.model_ids, st.slos, M)
        batch = E.Batch(eng, [dw], table, packed, COUNTS, options=dict(window_lanes=64, segment_requests=span))
        assert batch.kernel_name().count(",") == 6 and pcs
        batch.run()
        batch.sync()
        out = batch.fetch()
        batch.close()
        assert_batch_matches(out, oracle_batch(st, table, packed), 0, packed[0], where=f"uneven {uneven}")
        dw.close()


@pytest.mark.parametrize("faster,cut", [(1.0, True), (60.0, False)])
def test_streams_that_overload_the_groups_are_not_cut(faster, cut):
    """Several groups for every model and far more requests than they can take: the same results, one wavefront to a simulation."""
    eng = E.Engine.default()
    profiles, sols = _problem(3, (1, 2, 4), True, 9, 6, 12, 4)
    table = E.LatencyTable(profiles, [1])
    packed = E.pack_placements(sols, table)
    st = _with_pauses(11, 12000, 9, 0.8, 120)
    st.tstamps = st.tstamps / faster
    dw = E.DeviceWorkload(eng, st.tstamps, st.model_ids, st.slos, 9)
    batch = E.Batch(eng, [dw], table, packed, COUNTS)
    assert (batch.kernel_name().count(",") == 6) == cut
    batch.run()
    batch.sync()
    out = batch.fetch()
    batch.close()
    assert_batch_matches(out, oracle_batch(st, table, packed), 0, packed[0], where=f"faster {faster}")
    dw.close()


@pytest.mark.parametrize("bursty", [False, True])
@pytest.mark.parametrize("batching", [0, _lib.BATCHING])
def test_where_runs_would_not_agree_simulations_are_not_cut(batching, bursty):
    """Four groups for every model that are half busy (three quarters with batching): cut where arrivals come in bursts, not where they come evenly (a request
    each time goes to another group then, and runs that once chose differently go on doing so)."""
    eng = E.Engine.default()
    rng = np.random.default_rng(8)
    M, R, sizes = 9, 12000, [1, 2, 4, 8] if batching else [1]
    profiles, _ = _problem(8, (1,), True, M, 1, 1, 1)
    for p in profiles:
        for d in p.para_dict.values():
            for b in sizes[1:]:
                d.latency[b] = [x * (1 + 0.15 * (b - 1)) for x in d.latency[1]]
    sols = [ModelPlacement([ParallelConfig(1, 1, 1)] * 6, [[int(x) for x in rng.choice(M, 6, replace=False)] for _ in range(6)]) for _ in range(12)]
    table = E.LatencyTable(profiles, sizes)
    packed = E.pack_placements(sols, table)
    gaps = rng.gamma(1 / 64, 64, R) if bursty else rng.exponential(1.0, R)
    times = np.cumsum(gaps * (R / gaps.sum() / (25.0 if batching else 15.0)))       # a second, of the 34 that six groups can do
    ids, slos = rng.integers(0, M, R).astype(np.int32), rng.uniform(0.1, 0.8, R).astype(np.float32)
    dw = E.DeviceWorkload(eng, times, ids, slos, M)
    batch = E.Batch(eng, [dw], table, packed, batching)
    assert (batch.kernel_name().count(",") == (4 if batching else 6)) == bursty
    batch.run()
    batch.sync()
    out = batch.fetch()
    batch.close()
    dw.close()
    ref = oracle_batch(SimpleNamespace(tstamps=times, model_ids=ids, slos=slos), table, packed, batching=bool(batching))
    assert np.array_equal(out["n_good"][0], ref["n_good"])
    assert np.allclose(out["latency_sum"][0], ref["latency_sum"], rtol=1.4e-12 if batching else 0, atol=0)     # (12000 * 2^-53, as above)


@pytest.mark.parametrize("depths,uniform,groups,hosts,M", [((1,), True, 6, 7, 9), ((1, 2, 4), True, 6, 8, 9), ((1, 3, 5), False, 12, 9, 70)])
def test_runs_of_the_batching_simulator_taken_up_again(depths, uniform, groups, hosts, M):
    """As test_runs_taken_up_again_meet_others; latency sums within the bound above (25600 requests: 2.9e-12)."""
    eng = E.Engine.default()
    span, sizes = 512, [1, 2, 4, 8]
    streams = [_busy_between(51 + k, 300 * 64 + 17, M, 12.0, 60 * 64, 170 * 64) for k in range(2)] + [_busy_between(53, 400 * 64, M, 12.0, 40 * 64, 130 * 64)]
    late = _busy_between(54, 400 * 64, M, 12.0, 200 * 64, 290 * 64)
    gaps = np.diff(streams[2].tstamps, prepend=0.0)
    gaps[180 * 64:] = np.diff(late.tstamps, prepend=0.0)[180 * 64:]
    streams[2].tstamps = np.cumsum(gaps)
    dws = [E.DeviceWorkload(eng, s.tstamps, s.model_ids, s.slos, M) for s in streams]
    for B, flags in ((24, COUNTS), (40, 0)):
        profiles, sols = _problem(B + sum(depths), depths, uniform, M, groups, B, hosts)
        for p in profiles:
            for d in p.para_dict.values():
                for b in sizes[1:]:
                    d.latency[b] = [x * (1 + 0.15 * (b - 1)) for x in d.latency[1]]
        table = E.LatencyTable(profiles, sizes)
        packed = E.pack_placements(sols, table)
        batch = E.Batch(eng, dws, table, packed, flags | _lib.BATCHING, options=dict(segment_requests=span))
        assert batch.kernel_name().count(",") == 4            # (the last one: cut into runs)
        outs = []
        for _ in range(3):
            batch.run()
            batch.sync()
            assert batch.info()["runs_met_again"] > 0
            outs.append(batch.fetch())
        batch.close()
        for k, st in enumerate(streams):
            ref = oracle_batch(st, table, packed, batching=True)
            for out in outs:
                assert not out["status"].any() and np.array_equal(out["n_good"][k], ref["n_good"]), (B, k)
                for key in ("model_num_good", "group_num_requests", "group_num_good") if flags else ():
                    assert np.array_equal(out[key][k], ref[key]), (B, k, key)
                assert np.allclose(out["latency_sum"][k], ref["latency_sum"], rtol=3e-12, atol=0), (B, k)
                assert np.array_equal(out["latency_sum"][k], outs[0]["latency_sum"][k]), (B, k)
    for dw in dws:
        dw.close()


def test_where_simulations_of_the_batching_simulator_are_cut_by_themselves():
    """Few simulations of long streams, on every stream and paired; not with per-request outputs, and not short streams."""
    eng = E.Engine.default()
    M, sizes = 9, [1, 2, 4, 8]
    profiles, sols = _problem(3, (1, 2, 4), True, M, 6, 12, 4)
    for p in profiles:
        for d in p.para_dict.values():
            for b in sizes[1:]:
                d.latency[b] = [x * (1 + 0.15 * (b - 1)) for x in d.latency[1]]
    table = E.LatencyTable(profiles, sizes)
    packed = E.pack_placements(sols, table)
    streams = [_with_pauses(11, 20000, M, 0.8, 120), _with_pauses(12, 9000, M, 0.8, 120)]
    for s in streams:
        s.slos = np.where(np.isfinite(s.slos), s.slos, np.float32(0.4))
    dws = [E.DeviceWorkload(eng, s.tstamps, s.model_ids, s.slos, M) for s in streams]
    refs = [oracle_batch(s, table, packed, batching=True) for s in streams]
    for flags in (0, COUNTS):
        batch = E.Batch(eng, dws, table, packed, flags | _lib.BATCHING)
        assert batch.kernel_name().count(",") == 4            # (the last one: cut into runs)
        batch.run()
        batch.sync()
        out = batch.fetch()
        batch.close()
        for k in range(2):
            assert np.array_equal(out["n_good"][k], refs[k]["n_good"])
            assert np.allclose(out["latency_sum"][k], refs[k]["latency_sum"], rtol=3e-12, atol=0)     # (20000 requests, see above)
            for key in ("model_num_good", "group_num_requests", "group_num_good") if flags else ():
                assert np.array_equal(out[key][k], refs[k][key]), key
    of = np.arange(len(sols)) % 2
    got = E.eval_pairs(eng, dws, table, packed, of, COUNTS | _lib.BATCHING)
    for key in ("n_good", "model_num_good", "group_num_requests", "group_num_good"):
        assert np.array_equal(got[key], np.where((of == 0).reshape((-1,) + (1,) * (refs[0][key].ndim - 1)), refs[0][key], refs[1][key])), key
    for loads, flags in ((dws, COUNTS | _lib.WANT_PER_REQUEST), ([E.DeviceWorkload(eng, streams[0].tstamps[:7616], streams[0].model_ids[:7616], streams[0].slos[:7616], M)], 0)):
        batch = E.Batch(eng, loads, table, packed, flags | _lib.BATCHING)
        assert batch.kernel_name().count(",") == 3
        batch.close()
    for dw in dws:
        dw.close()


def _hip():
    """The HIP runtime that the library runs on (torch brings another one)."""
    with open("/proc/self/maps") as f:
        return C.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))


def _free_bytes():
    free, total = C.c_size_t(), C.c_size_t()
    assert _hip().hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@contextmanager
def _no_more_free_than(most):
    taken = []
    try:
        while _free_bytes() > most + (16 << 20) and len(taken) < 8:        # (of a large piece the runtime takes less than asked for)
            taken.append(C.c_void_p())
            assert _hip().hipMalloc(C.byref(taken[-1]), C.c_size_t(_free_bytes() - most)) == 0
        yield
    finally:
        for p in taken:
            assert _hip().hipFree(p) == 0


def test_batches_share_the_memory_of_their_runs():
    """The runs of a batch that is kept are in memory of the context: three batches hold as much of it as the largest, they may be run
    in any order, and what one call needed beyond 2 GiB is given back."""
    eng = E.Engine(0)                                     # (no memory of other tests' runs)
    profiles, sols = _problem(3, (1, 2, 4), True, 9, 6, 200, 4)
    table = E.LatencyTable(profiles, [1])
    st = _with_pauses(71, 60000, 9, 0.8, 120)
    dw = E.DeviceWorkload(eng, st.tstamps, st.model_ids, st.slos, 9)
    packed = [E.pack_placements(sols[:n], table) for n in (60, 200, 120)]
    refs = [oracle_batch(st, table, p) for p in packed]
    before = _free_bytes()
    batches = [E.Batch(eng, [dw], table, p, COUNTS) for p in packed]
    for b in batches:
        assert b.kernel_name().count(",") == 6            # (the last one: cut into runs)
    for k in (0, 1, 2, 0, 1):
        batches[k].run()
    for k in (0, 1, 2):
        assert_batch_matches(batches[k].fetch(), refs[k], 0, packed[k][0], where=f"batch {k}")
    # 200 simulations of 16 runs of 59 blocks, which may go on for 48: 15 * 107 * 64 values each (164 MB), marks and ends 36 MB
    assert before - _free_bytes() < 240 << 20
    for b in batches:
        b.close()
    dw.close()
    eng.close()


def test_simulations_are_not_cut_where_there_is_no_memory_for_their_runs():
    eng = E.Engine(0)
    profiles, sols = _problem(3, (1, 2, 4), True, 9, 6, 300, 4)
    table = E.LatencyTable(profiles, [1])
    st = _with_pauses(71, 60000, 9, 0.8, 120)
    dw = E.DeviceWorkload(eng, st.tstamps, st.model_ids, st.slos, 9)
    packed = E.pack_placements(sols, table)
    ref = oracle_batch(st, table, packed)
    batch = E.Batch(eng, [dw], table, packed, COUNTS)
    assert batch.kernel_name().count(",") == 6
    with _no_more_free_than(400 << 20):                   # (a quarter of that: 100 MiB)
        late = E.Batch(eng, [dw], table, packed, COUNTS)
        assert late.kernel_name().count(",") == 5
        for b in (batch, late):
            b.run()
            b.sync()
            assert b.kernel_name().count(",") == 5
            assert_batch_matches(b.fetch(), ref, 0, packed[0])
            b.close()
    dw.close()
    eng.close()


def test_batching_simulations_are_not_cut_where_there_is_no_memory_for_their_runs():
    """Marks and ends of 3200 runs of 400 models, 146 MB, do not fit into 120 MB."""
    eng = E.Engine(0)
    M, sizes = 400, [1, 2, 4, 8]
    profiles, sols = _problem(3, (1, 2, 4), True, M, 6, 64, 40)
    for p in profiles:
        for d in p.para_dict.values():
            for b in sizes[1:]:
                d.latency[b] = [x * (1 + 0.15 * (b - 1)) for x in d.latency[1]]
    table = E.LatencyTable(profiles, sizes)
    st = _with_pauses(71, 66000, M, 0.8, 120)
    st.slos = np.where(np.isfinite(st.slos), st.slos, np.float32(0.4))
    dw = E.DeviceWorkload(eng, st.tstamps, st.model_ids, st.slos, M)
    packed = E.pack_placements(sols, table)
    others = E.DeviceWorkload(E.Engine.default(), st.tstamps, st.model_ids, st.slos, M)
    ref = E.eval_batch(E.Engine.default(), [others], table, packed, _lib.BATCHING)        # (cut: the oracle takes ten seconds)
    others.close()
    batch = E.Batch(eng, [dw], table, packed, _lib.BATCHING)
    assert batch.kernel_name().count(",") == 4
    with _no_more_free_than(120 << 20):
        late = E.Batch(eng, [dw], table, packed, _lib.BATCHING)
        assert late.kernel_name().count(",") == 3
        for b in (batch, late):
            b.run()
            b.sync()
            assert b.kernel_name().count(",") == 3
            out = b.fetch()
            assert np.array_equal(out["n_good"], ref["n_good"])
            assert np.allclose(out["latency_sum"], ref["latency_sum"], rtol=8e-12, atol=0)      # (66000 requests, see above)
            b.close()
    dw.close()
    eng.close()
