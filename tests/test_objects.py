"""Placements and requests as flat arrays: the native reading of plain lists, tuples, ints and floats against the general code
that takes any other sequence, on the same values."""
from types import SimpleNamespace

import numpy as np
import pytest

from mms_amd import _objects, engine as E
from mms_amd.placement_policy import ModelPlacement
from mms_amd.profiling import ParallelConfig
from mms_amd.simulator.workload import Request


class Rows(list):
    """No plain list: the general code's."""


def _table(models):
    return E.LatencyTable([SimpleNamespace(para_dict={})] * models)


@pytest.mark.parametrize("row", [list, tuple])
@pytest.mark.parametrize("B,groups,models", [(0, 1, 3), (1, 0, 3), (1, 1, 1), (7, 5, 300), (65, 9, 20), (40, 70, 256)])
def test_placements(B, groups, models, row):
    rng = np.random.default_rng(B + groups)
    pcs = [ParallelConfig(1, int(o), int(p)) for o in (1, 2, 4) for p in (1, 2, 3, 8)]
    again = [ParallelConfig(*c) for c in pcs]        # equal configurations that are other objects
    sols = []
    for b in range(B):
        n = int(rng.integers(0, groups + 1)) if b else groups
        sols.append(ModelPlacement(row((pcs, again)[int(rng.integers(2))][int(rng.integers(12))] for _ in range(n)),
                                   row(row(int(m) for m in rng.integers(0, models, int(rng.integers(0, 6)))) for _ in range(n))))
    general = [ModelPlacement(s.group_configs, Rows(s.group_models)) for s in sols]
    tables = _table(models), _table(models)
    got, want = E.pack_placements(row(sols), tables[0]), E.pack_placements(general, tables[1])
    assert _objects.pack(general, {}, None) is None or B == 0
    assert tables[0].index == tables[1].index and tables[0].configs == tables[1].configs
    for g, w in zip(got, want):
        assert g.dtype == w.dtype and g.shape == w.shape and np.array_equal(g, w) and g.flags.writeable
    assert np.array_equal(E.count_models(sols), E.count_models(general)) and E.count_models(sols).dtype == np.int64
    if B > 1:       # every configuration is known now: the same ids without one being added
        assert np.array_equal(E.pack_placements(sols, tables[0])[1], want[1]) and len(tables[0].configs) == len(tables[1].configs)


@pytest.mark.parametrize("ids", [[np.int32(1), 2], [True, 0], [-1, 3], [2 ** 31 - 1, -2 ** 31], range(3)])
def test_ids_that_the_library_looks_at(ids):
    """What is no int or no id goes on as it did: the values reach the library, which refuses those outside 0..M-1."""
    sols = [ModelPlacement([ParallelConfig(1, 1, 1)], [ids])]
    assert E.pack_placements(sols, _table(300))[3].tolist() == [int(x) for x in ids]


@pytest.mark.parametrize("sol,error", [
    (ModelPlacement([ParallelConfig(1, 1, 1)], [[2 ** 31]]), OverflowError), (ModelPlacement([ParallelConfig(1, 1, 1)], [["a"]]), ValueError),
    (ModelPlacement([ParallelConfig(1, 1, 1)], []), ValueError), (ModelPlacement([[1]], [[0]]), TypeError), (object(), AttributeError)])
def test_placements_that_are_refused(sol, error):
    with pytest.raises(error):
        E.pack_placements([sol], _table(300))


def test_requests():
    names = {f"m{m}": m for m in range(5)}
    slos = [0.1, 1 / 3, float("inf"), 0.0, 5e-46, 1e-40, -1.0, 3.4028234e38, float("nan")]
    plain = [Request(f"m{k % 7}", None, s, k, {}) for k, s in enumerate(slos)]
    odd = plain + [Request("m1", None, s, 0, {}) for s in (None, 2, np.float32(0.3), np.float64(0.3))]
    for reqs in (plain, tuple(plain), [], odd, Rows(plain)):
        ids, got = E.request_arrays(reqs, names)
        assert ids.dtype == np.int32 and got.dtype == np.float32
        assert np.array_equal(ids, np.array([names.get(r.model_name, -1) for r in reqs], np.int32))
        assert np.array_equal(got, np.array([r.slo for r in reqs], np.float32), equal_nan=True)
    assert _objects.request_arrays(odd, names) is None and _objects.request_arrays(plain, names) is not None
    with pytest.raises(AttributeError):
        E.request_arrays([object()], names)
