"""Batched MatMul on bf16 parts, and MatMul operands read transposed in place
of a Transpose node, against 64-bit products.

|error| <= (K / 8 + 16) * 2^-24 * sum |a b|, as for the convolutions on parts.
"""

from __future__ import annotations

import numpy as np
import pytest

from spinnv2_amd.runtime import Model
from spinnv2_amd.spk import models, write_spk
from spinnv2_amd.spk.graph import Graph

from .helpers import rng_inputs, run_gpu

pytestmark = pytest.mark.gpu


def _close(got, a, b):
    a, b = a.astype(np.float64), b.astype(np.float64)
    want, size = a @ b, np.abs(a) @ np.abs(b)
    assert np.all(np.abs(got.reshape(want.shape) - want) <= (a.shape[-1] / 8 + 16) * 2.0 ** -24 * size)


# tiles' edges and remainders in M, N and K, on 64- and 32-row tiles
@pytest.mark.parametrize("batch,m,n,k", [(70, 1, 1, 3), (64, 64, 64, 32), (16, 65, 127, 33), (70, 33, 66, 70),
                                         (9, 129, 200, 31), (64, 31, 63, 130), (3, 400, 257, 101), (80, 5, 7, 64)])
def test_matmul_parts(gpu, batch, m, n, k):
    g = models.matmul_op([batch, m, k], [batch, k, n])
    xs = rng_inputs(g)
    with Model(write_spk(g, "mi355x")) as mdl:
        got = mdl(*xs)
        assert "matmul_parts" in mdl.kernel_name(0)
    _close(got, *xs)


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("k", [1, 2, 3])
def test_few_products(gpu, k, transposed):
    """One or two products are summed without parts, whose left-out products
    and extra roundings they would show: each product of K multiply-adds is
    rounded at most K times, so |error| <= K 2^-24 sum |a b|."""
    g = Graph("few")
    a, b = g.input("a", [64, 96, k]), g.input("b", [64, 96, k] if transposed else [64, k, 96])
    g.mark_output(g.matmul(a, g.transpose(g.add(b, b), [0, 2, 1]) if transposed else b))
    xs = rng_inputs(g)
    with Model(write_spk(g, "mi355x")) as mdl:
        got = mdl(*xs)
        names = [mdl.kernel_name(i) for i in range(len(g.nodes))]
    assert any("matmul_parts" in s for s in names) == (k > 2), names
    assert any("transpose_elided" in s for s in names) == (transposed and k > 2), names
    x, y = (v.astype(np.float64) for v in (xs[0], 2 * np.swapaxes(xs[1], 1, 2) if transposed else xs[1]))
    assert np.all(np.abs(got.reshape(64, 96, 96) - x @ y) <= k * 2.0 ** -24 * (np.abs(x) @ np.abs(y)))


@pytest.mark.parametrize("ta,tb", [(True, False), (False, True), (True, True)])
@pytest.mark.parametrize("batch,m,n,k", [(2, 20, 33, 12), (6, 64, 65, 130), (1, 100, 40, 67), (70, 64, 64, 32)])
def test_transposed_operands(gpu, monkeypatch, batch, m, n, k, ta, tb):
    """Transposes feeding only the MatMul are not run; with the views off they
    are, and the results are the same bits."""
    g = Graph("mm")
    a = g.input("a", [batch, k, m] if ta else [batch, m, k])
    b = g.input("b", [batch, n, k] if tb else [batch, k, n])
    ga, gb = g.add(a, a), g.add(b, b)
    ma = g.transpose(ga, [0, 2, 1]) if ta else ga
    mb = g.transpose(gb, [0, 2, 1]) if tb else gb
    g.mark_output(g.add(g.matmul(ma, mb), g.weight("zero", np.zeros(1, np.float32))))
    xs = rng_inputs(g)
    blob = write_spk(g, "mi355x")
    with Model(blob) as mdl:
        got = [mdl(*xs), mdl(*xs)]
        names = [mdl.kernel_name(i) for i in range(len(g.nodes))]
    assert sum("transpose_elided" in s for s in names) == ta + tb, names
    assert any("matmul_parts" in s and (",ta" in s) == ta and (",tb" in s) == tb for s in names), names
    np.testing.assert_array_equal(got[0], got[1])
    xa, xb = (np.swapaxes(x, 1, 2) if t else x for x, t in zip(xs, (ta, tb)))
    _close(got[0], 2 * xa, 2 * xb)
    monkeypatch.setenv("SPKV2_CONCAT_VIEWS", "0")
    with Model(blob) as mdl:
        plain = mdl(*xs)
        pnames = [mdl.kernel_name(i) for i in range(len(g.nodes))]
    assert not any("elided" in s for s in pnames), pnames
    np.testing.assert_array_equal(plain, got[0])


def test_transposed_operand_with_a_fault_armed(gpu):
    """With a fault event armed (here on a node's later invocation, so that
    nothing flips) every node runs on its own tensors."""
    g = Graph("mm")
    a, b = g.input("a", [4, 40, 24]), g.input("b", [4, 40, 30])
    s = g.softmax(a, -1)
    g.mark_output(g.matmul(g.transpose(s, [0, 2, 1]), b))
    xs = rng_inputs(g)
    with Model(write_spk(g, "mi355x")) as mdl:
        one = mdl(*xs)
        assert mdl.set_fault_event({"node_id": 0, "tensor_id": g.nodes[0].outputs[0], "element_index": 0,
                                    "bit_index": 1, "invocation_index": 9, "enabled": 1}) == 0
        for i, x in enumerate(xs):
            mdl.set_input(i, x)
        mdl.run()
        two = mdl.get_output(0)
        assert not any("elided" in mdl.kernel_name(i) for i in range(len(g.nodes)))
    np.testing.assert_array_equal(two, one)


def test_matmul_special_values(gpu, monkeypatch):
    g = models.matmul_op([64, 40, 70], [64, 70, 50])
    xs = rng_inputs(g)
    xs[0][0, 1, 2], xs[0][1, 3, 4], xs[1][2, 5, 6] = np.inf, np.nan, np.float32(3.4e38)
    xs[0][3] *= 1e-36
    got = run_gpu(write_spk(g, "mi355x"), xs)[0].reshape(64, 40, 50)
    monkeypatch.setenv("SPKV2_MATMUL_KSPLIT", "0")
    want = run_gpu(write_spk(g, "mi355x"), xs)[0].reshape(64, 40, 50)
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(got[np.isinf(want)], want[np.isinf(want)])
    fin = np.isfinite(want)
    np.testing.assert_allclose(got[fin], want[fin], rtol=1e-4, atol=1e-4)
    np.testing.assert_allclose(got[3], want[3], rtol=1e-4, atol=1e-40)


@pytest.mark.parametrize("batch,size", [(64, 256), (1, 512)])
def test_matmul_special_values_cost(gpu, batch, size):
    """As for the layers: NaN in one matrix costs a few passes at most."""
    g = models.matmul_op([batch, size, size], [batch, size, size])
    xs = rng_inputs(g)
    odd = xs[0].copy()
    odd[0] = np.nan
    took = []
    with Model(write_spk(g, "mi355x")) as mdl:
        mdl.set_profiling(True)
        mdl.set_input(1, xs[1])
        for v in (xs[0], odd):
            mdl.set_input(0, v)
            mdl.run()
            assert "matmul_parts" in mdl.kernel_name(0)
            mdl.reset_node_times()
            for _ in range(5):
                mdl.run()
            took.append(mdl.node_time(0)[0])
    assert took[1] < 10 * took[0], took


@pytest.mark.parametrize("batch", [1, 64])  # 32- and 64-row tiles
@pytest.mark.parametrize("a_scale,b_scale", [(1e-37, 1.0), (1.0, 2e-38), (1e-41, 1e20), (1e12, 1e-36), (1e-43, 1e30),
                                             (1e33, 1e-30), (1e12, 1e16)])
def test_matmul_scaled_operands(gpu, batch, a_scale, b_scale):
    """As for the layers: operands near either end of the float range."""
    m, n, k = (512, 512, 70) if batch == 1 else (40, 50, 70)
    g = models.matmul_op([batch, m, k], [batch, k, n])
    a, b = ((x.astype(np.float64) * s).astype(np.float32) for x, s in zip(rng_inputs(g), (a_scale, b_scale)))
    with Model(write_spk(g, "mi355x")) as mdl:
        got = mdl(a, b).reshape(batch, m, n).astype(np.float64)
        assert "matmul_parts" in mdl.kernel_name(0)
    a, b = a.astype(np.float64), b.astype(np.float64)
    assert np.all(np.abs(got - a @ b) <= (k / 8 + 16) * 2.0 ** -24 * (np.abs(a) @ np.abs(b)) + 2.0 ** -150)
