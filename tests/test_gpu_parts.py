"""The implicit GEMM on bf16 parts (conv_split.hip) against 64-bit sums.

A float32 operand, scaled by 2^24, is the exact sum of three bf16 parts, and
the six largest of a product's nine part products are summed: the three left
out are below 2^-24 of the product together, and a sum of K products rounds
once per 16 of them and once per slice, so |error| <= (K / 8 + 16) * 2^-24 * sum |x w| with room
for the matrix core's own order within a step.
"""

from __future__ import annotations

import numpy as np
import pytest

from spinnv2_amd.spk import models, write_spk
from spinnv2_amd.spk.graph import Graph

from .helpers import FP32_TOL, rng_inputs, run_gpu, run_oracle, tnorm_err

pytestmark = pytest.mark.gpu

PARTS_CFGS = [27, 28, 29]  # 128x64, 64x64 and 32x128 tiles


def _force(monkeypatch, cfg, split=1):
    monkeypatch.setenv("SPKV2_CONV_TUNE", "0")
    monkeypatch.setenv("SPKV2_CONV_SMALLK", "0")
    monkeypatch.setenv("SPKV2_CONV_CFG", str(cfg))
    if split >= 1000:
        monkeypatch.setenv("SPKV2_CONV_HYBRID", str(split - 1000))
    else:
        monkeypatch.setenv("SPKV2_CONV_SPLITK", str(split))


def _columns(x, k, stride, pads):
    """[N, C*k*k, OH*OW] in float64, k ordered (c, kh, kw)."""
    t, l, b, r = pads
    x = np.pad(x.astype(np.float64), ((0, 0), (0, 0), (t, b), (l, r)))
    oh, ow = (x.shape[2] - k) // stride + 1, (x.shape[3] - k) // stride + 1
    cols = [x[:, :, i:i + (oh - 1) * stride + 1:stride, j:j + (ow - 1) * stride + 1:stride]
            for i in range(k) for j in range(k)]
    return np.stack(cols, axis=2).reshape(x.shape[0], -1, oh * ow)


def _check(got, g, xs, k, stride, pads):
    w = g.tensors[g.nodes[0].inputs[1]].data.astype(np.float64)
    b = g.tensors[g.nodes[0].inputs[2]].data.astype(np.float64)[None, :, None]
    cols = _columns(xs[0], k, stride, pads)
    w2 = w.reshape(w.shape[0], -1)
    want, size = w2 @ cols + b, np.abs(w2) @ np.abs(cols) + np.abs(b)
    if len(xs) > 1:
        r = xs[1].astype(np.float64).reshape(want.shape)
        want, size = want + r, size + np.abs(r)
    K = w2.shape[1]
    err = np.abs(got.reshape(want.shape).astype(np.float64) - want)
    assert np.all(err <= (K / 8 + 16) * 2.0 ** -24 * size), float(np.max(err / size) * 2 ** 24)
    return float(np.linalg.norm(err) / np.linalg.norm(want))


# (N, Cin, H, W, Cout, k, stride, pads, residual): tiles' edges and
# remainders in M (1 .. 129 rows), N (1 pixel .. several tiles) and K (3 .. 648)
CASES = [
    (1, 3, 1, 1, 1, 1, 1, [0, 0, 0, 0], False),
    (1, 31, 7, 9, 33, 1, 1, [0, 0, 0, 0], True),
    (3, 33, 8, 8, 64, 3, 1, [1, 1, 1, 1], False),
    (2, 72, 11, 13, 129, 3, 1, [1, 1, 1, 1], True),
    (2, 64, 16, 17, 128, 1, 2, [0, 0, 0, 0], False),
    (1, 16, 9, 21, 31, 3, 2, [0, 1, 1, 0], False),
    (2, 5, 23, 19, 40, 7, 2, [3, 3, 3, 3], False),
]


@pytest.mark.parametrize("split", [1, 3, 1002])
@pytest.mark.parametrize("cfg", PARTS_CFGS)
@pytest.mark.parametrize("case", CASES, ids=[f"case{i}" for i in range(len(CASES))])
def test_parts_conv(gpu, monkeypatch, case, cfg, split):
    n, c, h, w, m, k, s, pads, res = case
    _force(monkeypatch, cfg, split)
    g = models.single_conv(n, c, h, w, m, k, s, act=None, residual=res, pads=pads)
    xs = rng_inputs(g)
    for implicit in ("0", "1"):
        monkeypatch.setenv("SPKV2_IMPLICIT_PAD", implicit)
        _check(run_gpu(write_spk(g, "mi355x"), xs)[0], g, xs, k, s, pads)


@pytest.mark.parametrize("cfg", PARTS_CFGS)
def test_parts_hybrid_schedule(gpu, monkeypatch, cfg):
    """More tiles than CUs: whole tiles, then k slices of the rest."""
    _force(monkeypatch, cfg, 1004)
    g = models.single_conv(9, 160, 50, 50, 160, 1, act=None)
    xs = rng_inputs(g)
    _check(run_gpu(write_spk(g, "mi355x"), xs)[0], g, xs, 1, 1, [0, 0, 0, 0])


@pytest.mark.parametrize("trans_a", [0, 1])
@pytest.mark.parametrize("cfg", PARTS_CFGS)
@pytest.mark.parametrize("split", [1, 2])
@pytest.mark.parametrize("rows,k,m", [(5, 64, 10), (33, 36, 129), (130, 100, 64), (70, 37, 65), (65, 4, 33), (6, 3, 8),
                                      (129, 135, 132)])
def test_parts_gemm(gpu, monkeypatch, rows, k, m, cfg, split, trans_a):
    _force(monkeypatch, cfg, split)
    g = models.single_gemm(rows, k, m, trans_a=trans_a)
    xs = rng_inputs(g)
    a = xs[0].astype(np.float64).T if trans_a else xs[0].astype(np.float64)
    b, c = (g.tensors[t].data.astype(np.float64) for t in g.nodes[0].inputs[1:3])
    got = run_gpu(write_spk(g, "mi355x"), xs)[0].reshape(rows, m)
    assert np.all(np.abs(got - (a @ b + c)) <= (k / 8 + 16) * 2.0 ** -24 * (np.abs(a) @ np.abs(b) + np.abs(c)))


@pytest.mark.parametrize("cfg", [6, *PARTS_CFGS])
def test_gemm_rows_at_any_address(gpu, monkeypatch, cfg):
    """A caller's input one float past an aligned address, NaN around it."""
    from spinnv2_amd.runtime import DeviceBuffer, Model

    _force(monkeypatch, cfg, 2)
    rows, k, m = 67, 70, 36
    g = models.single_gemm(rows, k, m)
    x = rng_inputs(g)[0]
    whole = np.full(x.size + 9, np.nan, np.float32)
    whole[1:1 + x.size] = x.ravel()
    with Model(write_spk(g, "mi355x")) as mdl:
        buf = DeviceBuffer(whole.nbytes)
        buf.upload(whole)
        view = type("View", (), {"ptr": type(buf.ptr)(buf.ptr.value + 4), "nbytes": x.nbytes})
        mdl.bind_input(0, view)
        mdl.run()
        got = mdl.get_output(0).reshape(rows, m)
        buf.free()
    a = x.astype(np.float64)
    b, c = (g.tensors[t].data.astype(np.float64) for t in g.nodes[0].inputs[1:3])
    assert np.all(np.abs(got - (a @ b + c)) <= (k / 2 + 16) * 2.0 ** -24 * (np.abs(a) @ np.abs(b) + np.abs(c)))


@pytest.mark.parametrize("relu", [False, True])
@pytest.mark.parametrize("c,k", [(16, 1), (64, 1), (16, 3), (256, 1), (64, 3), (256, 3)])
def test_parts_error_is_below_the_fp32_tiles(gpu, monkeypatch, c, k, relu):
    """2-norm error against 64 bits, K = 16 to 2304: no larger than that of
    the fp32 MFMA tile it takes the place of."""
    g = models.single_conv(2, c, 12, 12, 96, k, 1, k // 2, act=None)
    xs = [np.maximum(x, 0) if relu else x for x in rng_inputs(g)]
    err = {}
    for cfg in (6, *PARTS_CFGS):
        _force(monkeypatch, cfg)
        err[cfg] = _check(run_gpu(write_spk(g, "mi355x"), xs)[0], g, xs, k, 1, [k // 2] * 4)
    print(err)
    assert all(err[p] <= err[6] for p in PARTS_CFGS), err


@pytest.mark.parametrize("cfg", PARTS_CFGS)
@pytest.mark.parametrize("c", [1, 2])
def test_few_products(gpu, monkeypatch, c, cfg):
    """Layers of one or two products an output keep float32 multiply-adds:
    |error| <= K 2^-24 sum |w x|."""
    _force(monkeypatch, cfg)
    g = models.single_conv(1, c, 64, 64, 128, 1, act=None, bias=False)
    xs = rng_inputs(g)
    w = g.tensors[g.nodes[0].inputs[1]].data.astype(np.float64).reshape(128, c)
    x = xs[0].astype(np.float64).reshape(c, -1)
    got = run_gpu(write_spk(g, "mi355x"), xs)[0].reshape(128, -1)
    assert np.all(np.abs(got - w @ x) <= c * 2.0 ** -24 * (np.abs(w) @ np.abs(x)))


@pytest.mark.parametrize("implicit", ["0", "1"])
@pytest.mark.parametrize("cfg", PARTS_CFGS)
def test_parts_special_values(gpu, monkeypatch, cfg, implicit):
    """Infinities, NaN, values next to the largest and the smallest floats
    give what the fp32 tile gives, and only where it does."""
    monkeypatch.setenv("SPKV2_IMPLICIT_PAD", implicit)
    rng = np.random.default_rng(3)
    w = rng.standard_normal((40, 32, 3, 3)).astype(np.float32)
    w[5, 3, 1, 1], w[6, 4, 0, 0] = np.inf, np.nan
    x = rng.standard_normal((2, 32, 10, 10)).astype(np.float32)
    x[0, 1, 2, 3], x[0, 2, 7, 7], x[1, 0, 0, 0] = np.inf, -np.inf, np.nan
    x[1, 5, 5, 5], x[1, 6, 8, 8] = np.float32(3.4e38), np.float32(1e-30)
    g = Graph("special")
    g.mark_output(g.conv(g.input("x", list(x.shape)), w, np.zeros(40, np.float32), pad=1))
    outs = []
    for c in (6, cfg):
        _force(monkeypatch, c)
        outs.append(run_gpu(write_spk(g, "mi355x"), [x])[0])
    want, got = outs
    np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
    np.testing.assert_array_equal(got[np.isinf(want)], want[np.isinf(want)])
    fin = np.isfinite(want)
    np.testing.assert_allclose(got[fin], want[fin], rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("cfg", PARTS_CFGS)
def test_parts_special_values_cost(gpu, monkeypatch, cfg):
    """A wave's block summed again runs about as many fp32 MFMA cycles as an
    fp32 tile, some three times the block's own: NaN may not cost a multiple
    of the number of outputs (a lane summing its own alone took 100 to 170
    times a whole pass)."""
    from spinnv2_amd.runtime import Model

    _force(monkeypatch, cfg)
    g = models.single_conv(16, 256, 14, 14, 256, 3, 1, 1, act=None)
    x = rng_inputs(g)[0]
    pixel, image = x.copy(), x.copy()
    pixel[3, 5, 7, 7], image[3] = np.nan, np.nan
    took = []
    with Model(write_spk(g, "mi355x")) as mdl:
        mdl.set_profiling(True)
        for v in (x, pixel, image):
            mdl.set_input(0, v)
            mdl.run()
            mdl.reset_node_times()
            for _ in range(5):
                mdl.run()
            took.append(mdl.node_time(0)[0])
    assert max(took[1:]) < 10 * took[0], took


@pytest.mark.parametrize("scale", [1e-36, 1e-30, 1e30])
def test_parts_scaled_inputs(gpu, monkeypatch, scale):
    """Inputs whose smaller parts would be denormal (1e-36), and far from 1."""
    _force(monkeypatch, 28)
    g = models.single_conv(1, 32, 6, 7, 40, 3, 1, 1, act=None, bias=False)
    xs = [(x * np.float64(scale)).astype(np.float32) for x in rng_inputs(g)]
    got = run_gpu(write_spk(g, "mi355x"), xs)[0].astype(np.float64).ravel()
    w = g.tensors[g.nodes[0].inputs[1]].data.astype(np.float64).reshape(40, -1)
    cols = _columns(xs[0], 3, 1, [1, 1, 1, 1])
    want, size = (w @ cols).ravel(), (np.abs(w) @ np.abs(cols)).ravel()
    assert np.all(np.abs(got - want) <= 288 * 2.0 ** -24 * size)


@pytest.mark.parametrize("cfg", PARTS_CFGS)
@pytest.mark.parametrize("w_scale,x_scale", [(1e-37, 1.0), (2e-38, 1.0), (1e-41, 1e20), (1e12, 1e-36), (1e20, 1e-38),
                                             (1e30, 1e-43), (1e-30, 1e33), (1e33, 1e-30), (1e16, 1e12)])
def test_parts_scaled_operands(gpu, monkeypatch, w_scale, x_scale, cfg):
    """Operands whose smaller parts would lie below the smallest bf16, and
    those that do not stay finite when scaled for the split (1e33, and sums of
    1e28): the bound of the other tests, and half of the smallest float."""
    _force(monkeypatch, cfg)
    rng = np.random.default_rng(9)
    w = (rng.standard_normal((40, 32, 3, 3)) * w_scale).astype(np.float32)
    x = (rng.standard_normal((1, 32, 6, 7)) * x_scale).astype(np.float32)
    g = Graph("scaled")
    g.mark_output(g.conv(g.input("x", list(x.shape)), w, np.zeros(40, np.float32), pad=1))
    cols, w2 = _columns(x, 3, 1, [1, 1, 1, 1])[0], w.astype(np.float64).reshape(40, -1)
    want, size = w2 @ cols, np.abs(w2) @ np.abs(cols)
    for implicit in ("0", "1"):
        monkeypatch.setenv("SPKV2_IMPLICIT_PAD", implicit)
        got = run_gpu(write_spk(g, "mi355x"), [x])[0].astype(np.float64).reshape(want.shape)
        err = np.abs(got - want)
        assert np.all(err <= (288 / 8 + 16) * 2.0 ** -24 * size + 2.0 ** -150), float(np.max(err / size) * 2 ** 24)


# (C, H, W, Cout, k, stride, pads, dilation, residual, activation): dilation,
# asymmetric padding, the most taps a side that the tap table holds and one more
IPAD_CASES = [
    (16, 13, 11, 40, 3, 1, [1, 1, 1, 1], 1, True, "Relu"),
    (8, 20, 20, 24, 3, 1, [2, 2, 2, 2], 2, True, None),
    (8, 21, 18, 70, 3, 2, [3, 0, 1, 5], 3, False, "Silu"),
    (3, 20, 17, 33, 5, 1, [8, 4, 0, 6], 2, False, "Relu"),
    (2, 19, 16, 33, 15, 1, [7, 7, 7, 7], 1, False, "Silu"),
    (2, 19, 18, 33, 16, 1, [8, 8, 7, 7], 1, False, "Relu"),
]


@pytest.mark.parametrize("implicit", ["1", "0"])
@pytest.mark.parametrize("cfg", PARTS_CFGS)
@pytest.mark.parametrize("case", IPAD_CASES, ids=[f"ipad{i}" for i in range(len(IPAD_CASES))])
def test_parts_implicit_padding(gpu, monkeypatch, case, cfg, implicit):
    from spinnv2_amd.runtime import Model

    _force(monkeypatch, cfg)
    monkeypatch.setenv("SPKV2_IMPLICIT_PAD", implicit)
    c, h, w, m, k, s, pads, d, res, act = case
    g = models.single_conv(2, c, h, w, m, k, s, dilation=d, act=act, residual=res, pads=pads)
    blob = write_spk(g, "mi355x")
    xs = rng_inputs(g)
    with Model(blob) as mdl:
        got = mdl(*xs)
        name = mdl.kernel_name(0)
    assert "conv_split_f32" in name, name
    assert (",ipad" in name) == (implicit == "1" and k <= 15), name
    assert tnorm_err(got, run_oracle(blob, xs)[0]) <= FP32_TOL


@pytest.mark.parametrize("split", [1, 2])
def test_parts_tiles_share_one_summation_order(gpu, monkeypatch, split):
    """As for the fp32 tiles: timing may choose among the tiles, and between a
    copy and checked taps, for the same cut of k."""
    g = models.single_conv(2, 64, 15, 14, 100, 3, 1, 1, act=None)
    xs = rng_inputs(g)
    outs = []
    for cfg in PARTS_CFGS:
        _force(monkeypatch, cfg, split)
        for implicit in ("0", "1"):
            monkeypatch.setenv("SPKV2_IMPLICIT_PAD", implicit)
            outs.append(run_gpu(write_spk(g, "mi355x"), xs)[0])
    for y in outs[1:]:
        np.testing.assert_array_equal(y.view(np.uint32), outs[0].view(np.uint32))
