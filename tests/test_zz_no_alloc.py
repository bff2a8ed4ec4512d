"""The entry point that allocates nothing, mmsim_eval_batch_static, against mmsim_eval_batch.

Both are called through the C ABI on the same inputs; every result array must be identical (the two
share the packing code and the kernels, only the home of the device buffers differs).  Two calls in a
row, the second with a smaller input, so that what the first call left in the static scratch would
show if anything that must start at zero were not cleared.  Collected last (file name): a failure
here must not hide the other tests.
"""
import json
import os
import subprocess
import sys

import numpy as np
import pytest

from mms_amd import _lib, engine as E
from mms_amd.synthetic import make_config

pytestmark = pytest.mark.gpu


def _same(a, b, where):
    assert a.keys() == b.keys(), where
    for k in a:
        if a[k].dtype.kind == "f":
            assert np.array_equal(a[k].view(np.uint64), b[k].view(np.uint64)), f"{k} differs {where}"
        else:
            assert np.array_equal(a[k], b[k]), f"{k} differs {where}"


def _both(eng, dws, table, packed, flags, where):
    print(f"no-alloc entry point: {where}, flags {flags}", flush=True)
    got = E.eval_batch(eng, dws, table, packed, flags, static=True)
    ref = E.eval_batch(eng, dws, table, packed, flags, static=False)
    _same(got, ref, where)
    return got


def test_static_entry_point_equals_the_allocating_one_on_two_calls_in_a_row():
    eng = E.Engine.default()
    counts = _lib.WANT_MODEL_COUNTS | _lib.WANT_GROUP_COUNTS
    # first call: configuration 2, all 64 placements x 2 seeds, counts and per-request outputs
    cfg = make_config(2, 64)
    table = E.LatencyTable(cfg.profiles, cfg.batch_sizes)
    streams = [cfg.stream(s) for s in cfg.base_seeds[:2]]
    dws = [E.DeviceWorkload(eng, s.tstamps[:3000], s.model_ids[:3000], s.slos[:3000], cfg.num_models)
           for s in streams]
    big = _both(eng, dws, table, E.pack_placements(cfg.placements, table), counts | _lib.WANT_PER_REQUEST,
                "cfg 2, 64 placements x 2 seeds x 3000 requests")
    assert big["n_good"].sum() > 0
    # second call, smaller: 9 placements x 1 seed x a shorter stream, counts only, then scores only
    few = E.pack_placements(cfg.placements[5:14], table)
    dw1 = [E.DeviceWorkload(eng, streams[0].tstamps[:700], streams[0].model_ids[:700],
                            streams[0].slos[:700], cfg.num_models)]
    small = _both(eng, dw1, table, few, counts, "cfg 2, 9 placements x 1 seed x 700 requests")
    assert small["n_good"].sum() > 0
    _both(eng, dw1, table, few, 0, "scores only")
    # the batching simulator shares the scratch
    cfg5 = make_config(5, 24)
    t5 = E.LatencyTable(cfg5.profiles, cfg5.batch_sizes)
    s5 = cfg5.stream(0)
    dw5 = [E.DeviceWorkload(eng, s5.tstamps[:2000], s5.model_ids[:2000], s5.slos[:2000], cfg5.num_models)]
    _both(eng, dw5, t5, E.pack_placements(cfg5.placements, t5), _lib.BATCHING | counts, "cfg 5, 24 placements, batching")
    # and the first input again: same answer as before
    again = E.eval_batch(eng, dws, table, E.pack_placements(cfg.placements, table),
                         counts | _lib.WANT_PER_REQUEST, static=True)
    _same(again, big, "first input again")


def test_static_entry_point_refuses_what_does_not_fit():
    eng = E.Engine.default()
    cfg = make_config(2, 64)
    table = E.LatencyTable(cfg.profiles, cfg.batch_sizes)
    st = cfg.stream(0)
    dw = [E.DeviceWorkload(eng, st.tstamps, st.model_ids, st.slos, cfg.num_models)]
    packed = E.pack_placements(cfg.placements, table)
    # per-request outputs of 512 placements x 9.6k requests: 512 * 9600 * 9 bytes = 44 MB, beyond the scratch
    with pytest.raises(_lib.MmsimError) as err:
        E.eval_batch(eng, dw, table, E.pack_placements(cfg.placements * 8, table), _lib.WANT_PER_REQUEST, static=True)
    assert err.value.code == _lib.E_NOMEM and str(_lib.STATIC_SCRATCH_BYTES) in str(err.value)
    # the scratch is usable afterwards
    got = E.eval_batch(eng, dw, table, packed, 0, static=True)
    ref = E.eval_batch(eng, dw, table, packed, 0, static=False)
    _same(got, ref, "after a refusal")


def test_static_entry_point_takes_large_batches_of_small_tables():
    """9900 placements of 100 models in eight-stage groups: the kernel with requests side by side takes them in 2 MB, the
    tables of the others would not fit the scratch beside their results."""
    from mms_amd.placement_policy.base_policy import ModelPlacement
    from mms_amd.profiling import ParallelConfig, synthetic_profile
    eng = E.Engine.default()
    M, pc = 100, ParallelConfig(1, 1, 8)
    table = E.LatencyTable([synthetic_profile(f"m{m}", 0.1 + 0.001 * m, [pc]) for m in range(M)], [1])
    rng = np.random.default_rng(1)
    sols = [ModelPlacement([pc, pc], [rng.choice(M, 5, replace=False).tolist() for _ in range(2)]) for _ in range(100)]
    packed = E.pack_placements([sols[b % 100] for b in range(9900)], table)
    dw = [E.DeviceWorkload(eng, np.cumsum(rng.exponential(0.002, 500)), rng.integers(0, M, 500).astype(np.int32),
                           np.full(500, 0.5, np.float32), M)]
    got = E.eval_batch(eng, dw, table, packed, 0, static=True)
    _same(got, E.eval_batch(eng, dw, table, packed, 0), "100 models")
    _same({k: v[:, :100] for k, v in got.items()}, E.eval_batch(eng, dw, table, E.pack_placements(sols, table)), "the first hundred")


_COUNT = """
import ctypes, json, sys
counter = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)      # before the library, so that its calls come here
counter.allocator_calls.restype = ctypes.c_long
from mms_amd import _lib, engine as E
from mms_amd.synthetic import make_config
eng = E.Engine.default()
cfg = make_config(2, 64)
table = E.LatencyTable(cfg.profiles, cfg.batch_sizes)
st = cfg.stream(0)
dw = [E.DeviceWorkload(eng, st.tstamps[:900], st.model_ids[:900], st.slos[:900], cfg.num_models)]
packed = E.pack_placements(cfg.placements, table)
def calls(static, flags):
    before = counter.allocator_calls()
    E.eval_batch(eng, dw, table, packed, flags, static=static)
    return counter.allocator_calls() - before
every = _lib.WANT_MODEL_COUNTS | _lib.WANT_GROUP_COUNTS | _lib.WANT_PER_REQUEST
first = [calls(True, f) for f in (0, every)]
plain = calls(False, 0)
again = [calls(True, f) for f in (0, every)]
eng.set_options(window_lanes=-1)      # the kernels that take one request after the other
print(json.dumps([first, plain, again, [calls(True, f) for f in (0, every)], calls(False, 0)]))
"""


def test_static_entry_point_calls_no_allocator(tmp_path):
    """Neither device memory nor pinned host memory is allocated or freed inside the call, the context's first one
    included (a process of its own, in which the library's calls of the allocators are counted)."""
    here = os.path.dirname(os.path.abspath(__file__))
    lib = str(tmp_path / "alloc_counter.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", os.path.join(here, "alloc_counter.c"), "-o", lib, "-ldl"], check=True)
    out = subprocess.run([sys.executable, "-c", _COUNT, lib], cwd=os.path.dirname(here), capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr
    first, plain, again, one_by_one, plain2 = json.loads(out.stdout.splitlines()[-1])
    assert plain > 0 and plain2 > 0          # the count sees the ordinary entry point's
    assert first == again == one_by_one == [0, 0]
