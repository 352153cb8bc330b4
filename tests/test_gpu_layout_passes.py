"""The padding, quantizing and averaging passes at the sizes where their
splits of the work end: bit-exact against plain numpy (padding through a conv
that copies its input; the INT8 passes through the oracle)."""

from __future__ import annotations

import numpy as np
import pytest

from spinnv2_amd.spk import models, write_spk
from spinnv2_amd.spk.graph import Graph
from spinnv2_amd.spk.passes import run_default_pipeline
from spinnv2_amd.spk.quantize import quantize_graph, quantize_int8_activations

from .helpers import rng_inputs, run_gpu, run_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,c,h,w,pads", [(1, 1, 1, 1, [1, 1, 1, 1]), (1, 2, 5, 3, [0, 1, 2, 0]), (3, 5, 7, 9, [1, 1, 1, 1]),
                                          (2, 33, 14, 14, [1, 1, 1, 1]), (2, 17, 31, 2, [2, 0, 0, 1])])
def test_padded_copy(gpu, monkeypatch, n, c, h, w, pads):
    """A conv whose one nonzero tap is a channel's corner reads the padded
    copy element for element."""
    monkeypatch.setenv("SPKV2_IMPLICIT_PAD", "0")
    monkeypatch.setenv("SPKV2_CONV_SMALLK", "0")
    x = models.make_input([n, c, h, w], 3)
    t, l, b, r = pads
    kh, kw = min(3, h + t + b), min(3, w + l + r)
    want = np.pad(x, ((0, 0), (0, 0), (t, b), (l, r)))
    for i, j in ((0, 0), (kh - 1, kw - 1)):
        wt = np.zeros((c, c, kh, kw), np.float32)
        wt[np.arange(c), np.arange(c), i, j] = 1
        g = Graph("pad")
        g.mark_output(g.conv(g.input("x", list(x.shape)), wt, np.zeros(c, np.float32), pad=pads))
        got = run_gpu(write_spk(g, "mi355x"), [x])[0].reshape(g.shape(g.outputs[0]))
        oh, ow = got.shape[2:]
        np.testing.assert_array_equal(got, want[:, :, i:i + oh, j:j + ow])


def _net(n, c, h, w, m):
    g = Graph("net")
    x = g.input("x", [n, c, h, w])
    p = np.random.default_rng(c * h + m)
    y = g.relu(g.conv(x, p.standard_normal((m, c, 1, 1)).astype(np.float32), np.zeros(m, np.float32)))
    return g, y


@pytest.mark.parametrize("n,c,h,w", [(1, 17, 3, 3), (2, 33, 8, 8), (1, 64, 5, 13), (3, 130, 7, 9), (1, 20, 1, 65)])
def test_int8_input_quantize(gpu, n, c, h, w):
    g, y = _net(n, c, h, w, 24)
    g.mark_output(y)
    run_default_pipeline(g)
    xs = rng_inputs(g)
    xs[0].ravel()[::7] *= 3.0
    blob = write_spk(g, "mi355x", quant_params=quantize_graph(g, [xs[0][:1]]))
    np.testing.assert_array_equal(run_gpu(blob, xs)[0], run_oracle(blob, xs)[0])


@pytest.mark.parametrize("n,c,h,w,m", [(1, 16, 1, 1, 8), (2, 20, 5, 7, 24), (1, 16, 9, 15, 64), (3, 32, 7, 7, 130),
                                       (2, 24, 17, 19, 256), (1, 16, 3, 86, 272)])
def test_int8_spatial_mean(gpu, n, c, h, w, m):
    g, y = _net(n, c, h, w, m)
    g.mark_output(g.flatten(g.reduce_mean(y, [2, 3], keepdims=1), 1))
    run_default_pipeline(g)
    xs = rng_inputs(g)
    blob = write_spk(g, "mi355x", quant_params=quantize_int8_activations(g, [xs[0]]))
    np.testing.assert_array_equal(run_gpu(blob, xs)[0], run_oracle(blob, xs)[0])
