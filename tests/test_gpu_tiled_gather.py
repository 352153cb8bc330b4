"""GatherElements that reads its indices through the Tile in front of it: the
oracle's bits, with the Tile elided and not, eager and as a graph."""

from __future__ import annotations

import numpy as np
import pytest

from spinnv2_amd.runtime import Model
from spinnv2_amd.spk import write_spk
from spinnv2_amd.spk.graph import Graph
from spinnv2_amd.spk.passes import run_default_pipeline

from .helpers import run_oracle

pytestmark = pytest.mark.gpu


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
        names = [m.kernel_name(node.id) for node in g.nodes]
        if views == "0" or second_reader:
            assert "tile_elided" not in names
        elif not between:
            assert "tile_elided" in names and "gather_elements<tiled>" in names
        m.close()
    for r in runs:
        for a, b in zip(r, runs[-1]):
            np.testing.assert_array_equal(a, b)
        picked = r[1].reshape(n, k, classes)
        np.testing.assert_allclose(picked, np.asarray(want[1]).reshape(n, k, classes), rtol=2e-6)
