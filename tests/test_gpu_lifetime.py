"""Contexts that end before what was made of them, as a garbage collector may have it."""
import pytest

from mms_amd import _lib, engine as E
from helpers import assert_batch_matches, oracle_batch
from test_gpu_window import COUNTS, _problem, _stream

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batching", [False, True])
def test_batches_and_workloads_outlive_their_context(batching):
    eng = E.Engine(0)
    profiles, sols = _problem(3, (1, 2), True, 9, 6, 20, 4)
    table = E.LatencyTable(profiles, [1])
    packed = E.pack_placements(sols, table)
    st = _stream(5, 9000, 9, 1.0)
    st.slos[st.slos > 1.0] = 0.5                          # (no infinite ones: the batching simulator refuses what they lead to)
    dw = E.DeviceWorkload(eng, st.tstamps, st.model_ids, st.slos, 9)
    batches = [E.Batch(eng, [dw], table, packed, COUNTS | (_lib.BATCHING if batching else 0)) for _ in range(2)]
    eng.close()
    for batch in batches:
        batch.run()
        batch.sync()
        out = batch.fetch()
        ref = oracle_batch(st, table, packed, batching=batching)
        if batching:
            assert (out["n_good"][0] == ref["n_good"]).all()
        else:
            assert_batch_matches(out, ref, 0, packed[0])
        batch.close()
    dw.close()
