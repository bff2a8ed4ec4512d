"""The plain simulator with requests side by side (sim_window.hip) against the CPU oracle, bit for bit: every number of
requests side by side, at the sizes where it can go wrong -- streams that end inside a block or a chunk of requests,
batches that do not fill a wavefront, models with more replicas than one and two fetches hold, depths that are powers of
two and others, tables with a latency per stage, infinite latencies and odd SLOs."""
from types import SimpleNamespace

import numpy as np
import pytest

from mms_amd import _lib, engine as E
from mms_amd.placement_policy.base_policy import ModelPlacement
from mms_amd.profiling import LatencyMemData, ParallelConfig, ProfilingResult
from oracle import oracle_c
from helpers import assert_batch_matches, oracle_batch

pytestmark = pytest.mark.gpu

COUNTS = _lib.WANT_MODEL_COUNTS | _lib.WANT_GROUP_COUNTS


def _problem(seed, depths, uniform, M, groups, B, hosts):
    rng = np.random.default_rng(seed)
    pcs = [ParallelConfig(1, 1, d) for d in depths]
    profiles = []
    for m in range(M):
        para = {}
        for pc in pcs:
            if rng.random() < 0.04:
                continue                                   # no profile: an infinite latency
            total = rng.uniform(0.05, 0.3)
            stages = np.full(pc.pp, total / pc.pp) if uniform else rng.dirichlet(np.ones(pc.pp)) * total
            para[pc] = LatencyMemData({1: [float(x) for x in stages]}, {1: [0.0] * pc.pp}, [1.0] * pc.pp)
        profiles.append(ProfilingResult(f"m{m}", para, 0, 0))
    sols = []
    for _ in range(B):
        n = int(rng.integers(1, groups + 1))
        sols.append(ModelPlacement([pcs[int(rng.integers(len(pcs)))] for _ in range(n)],
                                   [[int(x) for x in rng.choice(M, size=int(rng.integers(0, hosts + 1)), replace=False)] for _ in range(n)]))
    return profiles, sols


def _stream(seed, R, M, load):
    rng = np.random.default_rng(seed)
    gaps = rng.exponential(0.02 / load, size=R)
    gaps[rng.random(R) < 0.2] = 0.0
    ids = np.repeat(rng.integers(-1, M, R + 1), rng.geometric(0.4, R + 1))[:R].astype(np.int32)
    slos = rng.uniform(0.1, 0.8, R).astype(np.float32)
    slos[rng.random(R) < 0.02] = np.inf
    slos[rng.random(R) < 0.02] = np.nan
    return SimpleNamespace(tstamps=np.cumsum(gaps), model_ids=ids, slos=slos)


@pytest.mark.parametrize("lanes", [64, 32, 16, 8])
@pytest.mark.parametrize("depths,uniform,groups,hosts", [((1,), True, 6, 4), ((1,), True, 40, 5), ((1, 2, 4), True, 5, 4), ((1, 3, 4), False, 9, 5),
                                                        ((1, 2, 4, 8, 16), True, 7, 4), ((2, 5, 11), False, 12, 5), ((8, 32), True, 6, 4), ((7, 20), True, 6, 5)])
def test_requests_side_by_side(lanes, depths, uniform, groups, hosts):
    eng = E.Engine.default()
    M = 5 if groups > 6 else 9
    lengths = (0, 1, lanes - 1, lanes + 1, 127, 128, 1500)
    streams = [_stream(100 * lanes + k, R, M, 1.0 + k) for k, R in enumerate(lengths)]
    dws = [E.DeviceWorkload(eng, s.tstamps, s.model_ids, s.slos, M) for s in streams]
    for B, flags in ((1, COUNTS | _lib.WANT_PER_REQUEST), (64 // lanes + 1, COUNTS), (131, 0)):
        profiles, sols = _problem(B + sum(depths), depths, uniform, M, groups, B, hosts)
        table = E.LatencyTable(profiles, [1])
        packed = E.pack_placements(sols, table)
        batch = E.Batch(eng, dws, table, packed, flags, options=dict(window_lanes=lanes))
        assert batch.kernel_name().startswith(f"sim_window_kernel<{lanes},")
        for _ in range(2):                                 # a second run starts from scratch again
            batch.run()
            batch.sync()
        out = batch.fetch()
        batch.close()
        for k, st in enumerate(streams):
            ref = oracle_batch(st, table, packed, want_per_request=bool(flags & _lib.WANT_PER_REQUEST))
            if flags & _lib.WANT_PER_REQUEST:
                R = len(st.tstamps)
                assert np.array_equal(out["good"][k][:, :R], ref["good"]) and np.array_equal(out["finish"][k][:, :R], ref["finish"])
            assert_batch_matches(out, ref, k, packed[0], where=f"{lanes} lanes, B={B}, stream {k}")
    for dw in dws:
        dw.close()


@pytest.mark.parametrize("lanes", [64, 32, 16, 8])
@pytest.mark.parametrize("depths,uniform", [((1,), True), ((1, 2, 4), True), ((1, 3), False), ((2, 16), True)])
def test_where_the_number_of_replicas_changes_the_kernels_path(lanes, depths, uniform):
    """A block takes two, four, eight, sixteen or any number of groups per request, by its most listed model: placements with 2
    to 21 replicas of their most listed one, beside models with one, two or none; with more than eight wavefronts to a CU the
    kernel that keeps eight of them in registers, not sixteen."""
    eng = E.Engine.default()
    rng = np.random.default_rng(lanes + len(depths))
    counts = (2, 3, 4, 5, 7, 8, 9, 12, 13, 16, 17, 20, 21)
    profiles, _ = _problem(5, depths, uniform, 5, 1, 1, 1)
    pcs = [ParallelConfig(1, 1, d) for d in depths]
    sols = []
    for n in counts:
        hosts = [set() for _ in range(22)]
        for m, k in ((0, n), (1, 1), (2, 2), (3, max(1, n - 4))):      # (model 4: nowhere)
            for g in rng.permutation(22)[:k]:
                hosts[g].add(m)
        sols.append(ModelPlacement([pcs[min(int(rng.exponential(0.7)), len(pcs) - 1)] for _ in hosts], [sorted(int(m) for m in h) for h in hosts]))
    streams = [_stream(17 * lanes + k, R, 5, load) for k, (R, load) in enumerate(((lanes + 1, 4.0), (900, 2.0), (900, 9.0)))]
    table = E.LatencyTable(profiles)
    packed = E.pack_placements(sols, table)
    dws = [E.DeviceWorkload(eng, s.tstamps, s.model_ids, s.slos, 5) for s in streams]
    for flags, times in ((0, 1), (COUNTS, 1), (0, 60), (COUNTS, 60)):
        batch = E.Batch(eng, dws, table, E.pack_placements(sols * times, table), flags, options=dict(window_lanes=lanes))
        name = batch.kernel_name()
        assert name.startswith(f"sim_window_kernel<{lanes}, ") and name.split(", ")[3] == ("2" if lanes == 64 and times == 1 else "1")
        batch.run()
        batch.sync()
        out = batch.fetch()
        batch.close()
        for k, s in enumerate(streams):
            ref = oracle_batch(s, table, packed)
            for t in {0, times - 1}:
                mine = slice(t * len(sols), (t + 1) * len(sols))
                for key in ("n_good", "latency_sum") + (("model_num_good", "group_num_requests", "group_num_good") if flags else ()):
                    assert np.array_equal(out[key][k][mine], ref[key]), (k, t, key)
            assert k == 0 or 0 < ref["n_good"].min() and ref["n_good"].max() < len(s.tstamps)
    for dw in dws:
        dw.close()


def test_replaced_placements_and_the_kept_streams():
    """eval_pairs on this kernel (one placement to a wavefront), and a batch that outlives the workloads it was made from."""
    eng = E.Engine.default()
    profiles, sols = _problem(5, (1, 2, 4), True, 6, 5, 37, 4)
    table = E.LatencyTable(profiles, [1])
    packed = E.pack_placements(sols, table)
    streams = [_stream(40 + k, R, 6, 2.0) for k, R in enumerate((700, 1, 333))]
    dws = [E.DeviceWorkload(eng, s.tstamps, s.model_ids, s.slos, 6) for s in streams]
    of = np.arange(len(sols)) % 3
    got = E.eval_pairs(eng, dws, table, packed, of, COUNTS)
    batch = E.Batch(eng, dws, table, packed, COUNTS)
    for dw in dws:
        dw.close()
    batch.run()
    batch.sync()
    full = batch.fetch()
    batch.close()
    for k, st in enumerate(streams):
        ref = oracle_batch(st, table, packed)
        assert_batch_matches(full, ref, k, packed[0], where=f"stream {k}")
        mine = np.flatnonzero(of == k)
        for key in ("n_good", "latency_sum", "model_num_good", "group_num_requests"):
            assert np.array_equal(got[key][mine], full[key][k][mine]), key


@pytest.mark.parametrize("order", ["ascending", "descending", "repeated"])
def test_replica_tables_of_one_placement(order):
    """simulate_requests_mixed: tables whose rows list their groups in ascending order go through the requests side by
    side, others (another order decides ties, a group may be named twice) through the loop over requests."""
    eng = E.Engine.default()
    for seed in range(10):
        rng = np.random.default_rng(1000 + seed)
        M, G, R = int(rng.integers(1, 7)), int(rng.integers(1, 12)), (0, 1, 63, 64, 65, 500)[seed % 6]
        st = _stream(seed, R, M, 2.0)
        stages = rng.integers(1, 6, G).astype(np.int32)
        lat = np.zeros((M, G, int(stages.max())), np.float32)
        for g in range(G):
            lat[:, g, :stages[g]] = rng.uniform(0.01, 0.2, (M, stages[g]))
        m2g = np.full((M, G), -1, np.int32)
        for m in range(M):
            row = np.flatnonzero(rng.random(G) < 0.6)
            row = row[::-1] if order == "descending" else np.repeat(row, 2)[:G] if order == "repeated" else row
            m2g[m, :len(row)] = row
        fin, good = np.empty(R), np.empty(R, bool)
        counts = E.simulate_requests_mixed(eng, fin, good, st.tstamps, st.model_ids, st.slos, m2g, stages, lat)
        f0, g0, c0 = oracle_c.simulate_requests_mixed(st.tstamps, st.model_ids, st.slos, m2g, stages, lat)[:3]
        assert np.array_equal(good, g0) and np.array_equal(fin.view(np.uint64), f0.view(np.uint64)), seed
        for x, y in zip(counts, c0):
            assert np.array_equal(x, y), seed


def test_batches_beyond_the_lds_of_the_chip():
    """LDS holds the state of so many placements at once; more follow one another with one placement to a wavefront, and
    batches beyond 8192 go to the kernels that take one request after the other, with the same results; the next call is
    not affected."""
    eng = E.Engine.default()
    info = eng.device_info()
    M = 900
    profiles, sols = _problem(11, (1, 2), True, M, 3, 200, 6)
    table = E.LatencyTable(profiles, [1])
    st = _stream(7, 400, M, 3.0)
    dw = E.DeviceWorkload(eng, st.tstamps, st.model_ids, st.slos, M)
    # 32 bytes per model for the first four replicas and 4 for its groups, and some hundred bytes beside them
    at_least = info["lds_bytes_per_block"] // (36 * M + 600) * info["compute_units"]
    at_most = info["lds_bytes_per_block"] // (36 * M) * info["compute_units"]
    ref = oracle_batch(st, table, E.pack_placements(sols, table))
    for B, kernel in ((at_least, "sim_window_kernel<"), (at_most + 1, "sim_window_kernel<64,"), (8193, "sim_mixed_kernel<"),
                      (at_least, "sim_window_kernel<")):
        packed = E.pack_placements([sols[b % len(sols)] for b in range(B)], table)
        batch = E.Batch(eng, [dw], table, packed, 0)
        assert batch.kernel_name().startswith(kernel), (B, batch.kernel_name())
        batch.close()
        out = E.eval_batch(eng, [dw], table, packed)
        for key in ("n_good", "latency_sum"):
            assert np.array_equal(out[key][0], ref[key][np.arange(B) % len(sols)]), (B, key)
    dw.close()


@pytest.mark.parametrize("lanes", [64, 32, 16, 8])
def test_latency_tables_that_do_not_fit_beside_a_placement(lanes):
    """A table with a latency per stage, larger than LDS: the stage walk reads it from memory."""
    eng = E.Engine.default()
    M, depths = 80, tuple(range(1, 33))      # rows of 528 latencies and one more: 165 KB
    profiles, sols = _problem(lanes, depths, False, M, 7, 40, 12)
    table = E.LatencyTable(profiles, [1])
    for p in profiles:
        for pc in p.para_dict:
            table.config_id(pc)
    packed = E.pack_placements(sols, table)
    assert table.arrays()[0].shape[2] == 32 and 4 * M * (sum(depths) + 1) > eng.device_info()["lds_bytes_per_block"]
    streams = [_stream(60 + k, R, M, 4.0) for k, R in enumerate((1000, lanes + 1))]
    dws = [E.DeviceWorkload(eng, s.tstamps, s.model_ids, s.slos, M) for s in streams]
    for flags in (0, COUNTS):
        batch = E.Batch(eng, dws, table, packed, flags, options=dict(window_lanes=lanes))
        assert batch.kernel_name().endswith("false>") and batch.info()["lds_bytes"] < 4 * M * sum(depths)
        batch.run()
        batch.sync()
        out = batch.fetch()
        batch.close()
        for k, st in enumerate(streams):
            assert_batch_matches(out, oracle_batch(st, table, packed), k, packed[0], where=f"{lanes} lanes, stream {k}")
    for dw in dws:
        dw.close()


@pytest.mark.parametrize("stages,B,kernel", [(1, 4096, "window_kernel<64"), (1, 4097, "window_kernel<32"), (1, 8194, "window_kernel<16"),
                                            (1, 12288, "window_kernel<16"), (1, 12289, "mixed_kernel<"), (4, 3072, "window_kernel<64"),
                                            (4, 3073, "window_kernel<32"), (4, 6146, "window_kernel<16"), (4, 12288, "window_kernel<16"),
                                            (4, 12289, "mixed_kernel<"), (8, 8192, "window_kernel<16"), (8, 8193, "mixed_kernel<"),
                                            (16, 4096, "window_kernel<32"), (16, 4097, "mixed_kernel<"), (3, 12288, "window_kernel<16"),
                                            (32, 12288, "window_kernel<8"), (32, 12289, "mixed_kernel<")])
def test_which_batches_have_their_requests_side_by_side(stages, B, kernel):
    """The number of simulations and the depth of the groups decide (kernels of either side of every line)."""
    eng = E.Engine.default()
    profiles, sols = _problem(stages, (stages,), True, 4, 2, 64, 3)
    table = E.LatencyTable(profiles, [1])
    st = _stream(stages, 130, 4, 2.0)
    dw = E.DeviceWorkload(eng, st.tstamps, st.model_ids, st.slos, 4)
    of = np.arange(B) % len(sols)
    packed = E.pack_placements([sols[b] for b in of], table)
    batch = E.Batch(eng, [dw], table, packed, 0)
    assert batch.kernel_name().startswith("sim_" + kernel), batch.kernel_name()
    batch.run()
    batch.sync()
    out = batch.fetch()
    batch.close()
    once = E.eval_batch(eng, [dw], table, packed)      # (a batch for one call: what packing costs counts as well)
    dw.close()
    ref = oracle_batch(st, table, E.pack_placements(sols, table))
    for got in (out, once):
        assert np.array_equal(got["n_good"][0], ref["n_good"][of]) and np.array_equal(got["latency_sum"][0], ref["latency_sum"][of])


@pytest.mark.parametrize("B,R,pace,lanes", [(3073, 1024, 0.2, 64), (3073, 1023, 0.2, 32), (3073, 1024, 9.0, 32), (4096, 1100, 0.2, 64), (4097, 1100, 0.2, 32)])
def test_overloaded_streams_keep_the_widest_blocks(B, R, pace, lanes):
    """Streams that ask more than twice what the groups can do: 64 requests side by side up to four wavefronts to a SIMD."""
    eng = E.Engine.default()
    profiles, sols = _problem(4, (4,), True, 4, 2, 64, 3)
    table = E.LatencyTable(profiles, [1])
    st = _stream(4, R, 4, 2.0)
    st.tstamps *= pace
    dw = E.DeviceWorkload(eng, st.tstamps, st.model_ids, st.slos, 4)
    of = np.arange(B) % len(sols)
    batch = E.Batch(eng, [dw], table, E.pack_placements([sols[b] for b in of], table), 0)
    assert batch.kernel_name().startswith(f"sim_window_kernel<{lanes},"), batch.kernel_name()
    batch.run()
    batch.sync()
    out = batch.fetch()
    batch.close()
    dw.close()
    ref = oracle_batch(st, table, E.pack_placements(sols, table))
    assert np.array_equal(out["n_good"][0], ref["n_good"][of]) and np.array_equal(out["latency_sum"][0], ref["latency_sum"][of])
