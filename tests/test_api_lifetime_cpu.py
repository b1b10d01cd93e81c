"""The Python objects' C handles are destroyed adjoint, sim, context, each
once, whatever order the objects are finalized in."""
import itertools

import pytest

from demso_amd import api
from demso_amd import scene as sc


class Lib:
    """The C library's creating and destroying calls, recorded."""

    def __init__(self):
        self.made, self.gone = itertools.count(100), []

    def __getattr__(self, name):
        def call(*args):
            if name in ("dem_create", "dem_sim_create", "dem_adj_create"):
                args[0 if name == "dem_create" else -1]._obj.value = next(self.made)
            elif name in ("dem_destroy", "dem_sim_destroy", "dem_adj_destroy"):
                self.gone.append((name, args[0]))
            return 0

        return call


@pytest.fixture
def objects(monkeypatch):
    lib = Lib()
    monkeypatch.setattr(api._lib, "load", lambda: lib)
    ctx = api.Context()
    sim = api.Simulation(ctx, sc.column_collapse(cols=4, rows=4))
    return lib, ctx, sim, api.Adjoint(sim)


ORDER = [("dem_adj_destroy", 102), ("dem_sim_destroy", 101), ("dem_destroy", 100)]


@pytest.mark.parametrize("first", ["ctx", "sim", "adj"])
def test_any_order_of_finalizers(objects, first):
    lib, ctx, sim, adj = objects
    # what a collected cycle does: the weak references are cleared, then the
    # finalizers run, in any order
    ctx._sims.clear()
    sim._adjoints.clear()
    todo = {"ctx": ctx, "sim": sim, "adj": adj}
    for o in [todo.pop(first), *todo.values()]:
        o.__del__()
    names = [n for n, _ in lib.gone]
    assert sorted(lib.gone) == sorted(ORDER)
    assert names.index("dem_adj_destroy") < names.index("dem_sim_destroy") < names.index("dem_destroy")


def test_closing_in_and_out_of_order(objects):
    lib, ctx, sim, adj = objects
    ctx.close()
    assert lib.gone == ORDER and sim.handle is None and adj.handle is None
    adj.close()
    sim.close()
    ctx.close()
    assert lib.gone == ORDER
