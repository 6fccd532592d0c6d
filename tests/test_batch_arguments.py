"""The batch calls hand the native library arrays of one entry per box: lists
with fewer entries are refused before the call, longer ones and iterators
taken.  The library is a stub that notes what it is given."""
import types

import pytest

from cassandra_amd import abi
from cassandra_amd import engine as E
from cassandra_amd import systems as S


class _Lib:
    def __init__(self):
        self.calls = []

    def cass_nvt_run_device_batch(self, h, n, ids, rngs, opts, nsteps, ens, recs):
        self.calls.append((n, len(rngs), len(opts), len(ens)))
        return 0

    def cass_regrow_run_device(self, h, n, boxes, rngs, nsteps, ens, recs):
        self.calls.append((n, len(rngs), len(boxes), len(ens)))
        return 0


def _engine():
    eng = object.__new__(E.Engine)
    eng.lib, eng.h = _Lib(), None
    system = S.System([S.species_lj()], [1], [S.species_lj().ref_coords[None]], [20.0] * 3, 300.0)
    boxes = [types.SimpleNamespace(id=k, system=system, params_prob_translate=lambda: 1.0) for k in range(3)]
    return eng, boxes


def _run(eng, entry, boxes, rngs, energies, locates):
    if entry == "nvt":
        return eng.nvt_run_batch(boxes, rngs, 2, energies)
    return eng.regrow_run(boxes, 0, locates, rngs, 2, energies)


@pytest.mark.parametrize("entry,short", [("nvt", "rngs"), ("nvt", "energies"), ("regrow", "rngs"),
                                         ("regrow", "energies"), ("regrow", "locates")])
def test_fewer_entries_than_boxes_are_refused(entry, short):
    eng, boxes = _engine()
    n = {"rngs": 3, "energies": 3, "locates": 3, short: 1}
    with pytest.raises(ValueError, match=short):
        _run(eng, entry, boxes, [abi.CassRng() for _ in range(n["rngs"])], [{}] * n["energies"], [[0]] * n["locates"])
    assert eng.lib.calls == []


@pytest.mark.parametrize("entry", ["nvt", "regrow"])
@pytest.mark.parametrize("extra", [0, 2])
def test_arrays_cover_every_box(entry, extra):
    eng, boxes = _engine()
    rngs = [abi.CassRng() for _ in range(3 + extra)]
    out = _run(eng, entry, boxes, rngs, iter([{"total": 1.5}] * (3 + extra)), iter([[0]] * (3 + extra)))
    n, *sizes = eng.lib.calls[0]
    assert n == 3 and min(sizes) >= 3
    assert len(out) == 3 and all(o["final"]["total"] == 1.5 for o in out)
