"""GatherElements that reads its indices through the Tile in front of it: the
oracle's bits, with the Tile elided and not, eager and as a graph."""

from __future__ import annotations

import numpy as np
import pytest

from spinnv2_amd.runtime import Model
from spinnv2_amd.spk import write_spk
from spinnv2_amd.spk.graph import Graph
from spinnv2_amd.spk.passes import run_default_pipeline
from spinnv2_amd.spk.planner import plan_memory

from .helpers import run_oracle


def _writers_over_indices(g, gather):
    """Memory classes of what is written, between a Tile and the
    GatherElements that may read through it, over the Tile's input."""
    plan = plan_memory(g).entries
    tile = g.nodes[g.tensors[gather.inputs[1]].producer]
    x = plan[tile.inputs[0]]
    return [plan[o].memory_class for n in g.nodes if tile.id < n.id <= gather.id for o in n.outputs
            if plan[o].offset < x.offset + x.size and x.offset < plan[o].offset + plan[o].size]


def _elidable(g):
    """The Tiles that must not run, by node id: one reader, and the indices
    in place until it has read them."""
    return {g.tensors[n.inputs[1]].producer for n in g.nodes if n.op_type == "GatherElements"
            and g.tensors[n.inputs[1]].consumers == [n.id] and not _writers_over_indices(g, n)}


def _names_as_elidable(m, g, elidable):
    for n in g.nodes:
        if n.op_type == "Tile":
            assert m.kernel_name(n.id) == ("tile_elided" if n.id in elidable else "tile")
        elif n.op_type == "GatherElements":
            tiled = g.tensors[n.inputs[1]].producer in elidable
            assert m.kernel_name(n.id) == ("gather_elements<tiled>" if tiled else "gather_elements")


def _two_gathers(n, anchors, classes, k):
    """Boxes and class scores of the same top rows, each gathered through a
    Tile of its own; outputs where the planner puts them."""
    g = Graph("two")
    b = g.input("b", [n, anchors, 4])
    x = g.input("x", [n, anchors, classes])
    s = g.add(x, x)  # exact, so that the same rows are the top ones everywhere
    top, idx = g.topk(g.reduce_max(s, [2], keepdims=0), k, axis=1, largest=1)
    i = g.unsqueeze(idx, 2)
    boxes = g.gather_elements(b, g.tile(i, [1, 1, 4]), axis=1)
    picked = g.gather_elements(s, g.tile(i, [1, 1, classes]), axis=1)
    for t in (top, boxes, picked):
        g.mark_output(t)
    run_default_pipeline(g)
    return g


# (sizes, whether a graph output, and nothing else, lies over the indices)
TWO = [((1, 500, 3, 50), False), ((2, 500, 33, 50), True), ((4, 8400, 80, 300), True), ((7, 1200, 3, 100), True)]


@pytest.mark.parametrize("size,over", TWO)
def test_two_gathers_cases(size, over):
    g = _two_gathers(*size)
    classes = {c for n in g.nodes if n.op_type == "GatherElements" for c in _writers_over_indices(g, n)}
    assert classes == ({"OUTPUT"} if over else set())


def _detect(n, anchors, classes, k, second_reader, between):
    """Scores' row maxima -> TopK -> Unsqueeze -> Tile -> GatherElements, for
    the scores and (with its own Tile) their first four columns."""
    g = Graph("tiled")
    x = g.input("x", [n, anchors, classes])
    x2 = g.unary("Sigmoid", x)
    top, idx = g.topk(g.reduce_max(x2, [2], keepdims=0), k, axis=1, largest=1)
    i = g.unsqueeze(idx, 2)
    wide = g.tile(i, [1, 1, classes])
    if between:  # work that may be given the index tensor's place, before the gather
        noise = g.reduce_mean(g.add(x, x), [1], keepdims=1)
        noise = g.add(g.unary("Sigmoid", noise), noise)
    picked = g.gather_elements(x2, wide, axis=1)
    outs = [top, picked]
    if second_reader:
        outs.append(g.add(wide, wide))
    if between:
        outs.append(noise)
    for t in outs:
        g.mark_output(t)
    run_default_pipeline(g)
    return g


@pytest.mark.gpu
@pytest.mark.parametrize("size,over", TWO)
def test_two_gathers_through_tiles(gpu, size, over):
    n, anchors, classes, k = size
    g = _two_gathers(*size)
    blob = write_spk(g, "mi355x")
    r = np.random.default_rng(anchors)
    b = r.standard_normal((n, anchors, 4)).astype(np.float32)
    x = r.standard_normal((n, anchors, classes)).astype(np.float32)
    want = run_oracle(blob, [b, x])
    elidable = _elidable(g)
    assert len(elidable) == (1 if over else 2)
    m = Model(blob)
    for graph in (False, True):
        m.set_graph_mode(graph)
        for _ in range(3 if graph else 1):
            m.set_input(0, b)
            m.set_input(1, x)
            m.run()
            for o in range(3):
                np.testing.assert_array_equal(np.asarray(m.get_output(o)).ravel(), np.asarray(want[o]).ravel())
    _names_as_elidable(m, g, elidable)
    m.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n,anchors,classes,k", [(1, 7, 1, 3), (2, 130, 5, 17), (3, 257, 80, 100)])
@pytest.mark.parametrize("second_reader", [False, True])
@pytest.mark.parametrize("between", [False, True])
def test_gather_through_tile(gpu, monkeypatch, n, anchors, classes, k, second_reader, between):
    g = _detect(n, anchors, classes, k, second_reader, between)
    blob = write_spk(g, "mi355x")
    x = np.random.default_rng(anchors).standard_normal((n, anchors, classes)).astype(np.float32)
    want = run_oracle(blob, [x])
    runs = []
    for views in ("1", "0"):
        monkeypatch.setenv("SPKV2_CONCAT_VIEWS", views)
        m = Model(blob)
        for graph in (False, True):
            m.set_graph_mode(graph)
            for _ in range(3 if graph else 1):
                m.set_input(0, x)
                m.run()
                runs.append([np.array(m.get_output(o)) for o in range(len(g.outputs))])
        _names_as_elidable(m, g, set() if views == "0" else _elidable(g))
        m.close()
    for r in runs:
        for a, b in zip(r, runs[-1]):
            np.testing.assert_array_equal(a, b)
        picked = r[1].reshape(n, k, classes)
        np.testing.assert_allclose(picked, np.asarray(want[1]).reshape(n, k, classes), rtol=2e-6)
