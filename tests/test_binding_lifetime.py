"""The order in which the binding frees what a program made, against a library
that only records the calls (no GPU): states before their graph, graphs and
batches before their context, each once, whichever way they go.  A reference
cycle (an exception's traceback holds one) is the hard case: the collector
clears weak references before it finalizes, in no order of use."""
import gc

import pytest

from grudon_amd import api


class _Recorder:
    def __init__(self):
        self.calls, self.made = [], 0

    def _create(self, out):
        self.made += 1
        out._obj.value = self.made
        return 0

    def __getattr__(self, name):
        def call(*args):
            if name.endswith(("_create", "_create_typed", "_from_csr")):
                return self._create(args[-1])
            if name in ("grd_state_free", "grd_graph_free", "grd_batch_free", "grd_destroy"):
                self.calls.append((name, args[0].value))
            return 0
        return call


@pytest.fixture
def made(monkeypatch):
    L = _Recorder()
    monkeypatch.setattr(api, "lib", lambda: L)
    ctx = api.Context(0)  # 1
    G = api.Graph.from_csr(ctx, [0, 0], [])  # 2
    S, T = api.State(G, api.CC), api.State(G, api.PR)  # 3, 4
    B = api.Batch(ctx, [([0, 0], [])])  # 5
    return L, [ctx, G, S, T, B]


def _check(calls):
    assert sorted(v for _, v in calls) == [1, 2, 3, 4, 5]  # each once
    at = {v: i for i, (_, v) in enumerate(calls)}
    assert max(at[3], at[4]) < at[2] < at[1] and at[5] < at[1]
    assert dict((v, n) for n, v in calls) == {1: "grd_destroy", 2: "grd_graph_free", 3: "grd_state_free",
                                              4: "grd_state_free", 5: "grd_batch_free"}


@pytest.mark.parametrize("order", [[0, 1, 2, 3, 4], [4, 3, 2, 1, 0], [1, 4, 0, 3, 2]])
def test_collected_in_a_cycle(made, order):
    L, objs = made
    cycle = [objs[i] for i in order]
    cycle.append(cycle)
    del objs
    made[1].clear()
    del cycle
    gc.collect()
    _check(L.calls)


@pytest.mark.parametrize("order", [[0], [1, 0], [2, 1, 4, 0], [3, 0], [4, 1, 2, 0]])
def test_freed_by_hand_in_any_order(made, order):
    """What is freed with its graph or context is no longer usable, and freeing
    it again does nothing."""
    L, objs = made
    for i in order + [0, 1, 2, 3, 4]:
        (objs[i].close if i == 0 else objs[i].free)()
    _check(L.calls)
    assert all(o.h is None for o in objs)
