"""Tensors whose last bytes lie within 64 KB of 2 GiB, the most a tensor of the
conv kernels may hold: accesses that are to do nothing must lie past them."""

from __future__ import annotations

import numpy as np
import pytest

from spinnv2_amd.runtime import Model
from spinnv2_amd.spk import write_spk
from spinnv2_amd.spk.graph import Graph

pytestmark = pytest.mark.gpu

N, H, W = 2, 4080, 4112  # N * 16 * H * W * 4 = 2^31 - 2^15


def _values(shape, seed):
    base = np.random.default_rng(seed).standard_normal(1 << 20).astype(np.float32)
    return np.resize(base, shape)


@pytest.mark.parametrize("cfg", [8, 17, 28])  # 32-row, 16-row thin and 64-row tiles
def test_outputs_up_to_two_gib(gpu, monkeypatch, cfg):
    """Rows past the 16 outputs of a tile store nothing."""
    monkeypatch.setenv("SPKV2_CONV_TUNE", "0")
    monkeypatch.setenv("SPKV2_CONV_SMALLK", "0")
    monkeypatch.setenv("SPKV2_CONV_CFG", str(cfg))
    monkeypatch.setenv("SPKV2_CONV_SPLITK", "1")
    x = _values((N, 4, H, W), 1)
    w = np.random.default_rng(2).standard_normal((16, 4, 1, 1)).astype(np.float32)
    g = Graph("wide")
    g.mark_output(g.conv(g.input("x", list(x.shape)), w, np.full(16, 3, np.float32)))
    with Model(write_spk(g, "mi355x")) as mdl:
        mdl.set_input(0, x)
        mdl.run()
        assert "smallk" not in mdl.kernel_name(0), mdl.kernel_name(0)
        got = mdl.get_output(0).reshape(N, 16, H * W)
    for n in range(N):
        for m in range(16):
            want = np.tensordot(w[m, :, 0, 0], x[n].reshape(4, -1), axes=1) + np.float32(3)
            # 5 roundings a side of terms below sum |w x| + 3
            size = np.tensordot(np.abs(w[m, :, 0, 0]), np.abs(x[n].reshape(4, -1)), axes=1) + 3
            assert np.all(np.abs(got[n, m] - want) <= 10 * 2.0 ** -24 * size), (n, m)


@pytest.mark.parametrize("cfg", [6, 28])
def test_checked_taps_of_a_slice_near_two_gib(gpu, monkeypatch, cfg):
    """A padded conv over half of a Split whose Concat is nearly that large:
    the Concat has no views, since checked taps count from ahead of a slice and
    its extent, that added, has to stay below the offset that stands for none."""
    W = 4110  # the longest input a conv takes is 64 KB shorter
    monkeypatch.setenv("SPKV2_CONV_TUNE", "0")
    monkeypatch.setenv("SPKV2_CONV_CFG", str(cfg))
    monkeypatch.setenv("SPKV2_CONV_SPLITK", "1")
    monkeypatch.setenv("SPKV2_IMPLICIT_PAD", "1")
    monkeypatch.setenv("SPKV2_PAD_HANDOFF", "0")
    rng = np.random.default_rng(3)
    x = _values((N, 1, H, W), 4)
    wa, wb = (rng.standard_normal(s).astype(np.float32) for s in ((10, 1, 1, 1), (6, 5, 3, 3)))
    wc = rng.standard_normal((1, 16, 1, 1)).astype(np.float32)
    g = Graph("slice")
    a = g.conv(g.input("x", list(x.shape)), wa, np.zeros(10, np.float32))
    p, q = g.split(a, [5, 5], axis=1)
    r = g.conv(q, wb, np.zeros(6, np.float32), pad=1)
    g.mark_output(g.conv(g.concat([p, q, r], axis=1), wc, np.zeros(1, np.float32)))
    with Model(write_spk(g, "mi355x")) as mdl:
        mdl.set_input(0, x)
        mdl.run()
        names = [mdl.kernel_name(i) for i in range(len(g.nodes))]
        got = mdl.get_output(0).reshape(N, H, W)
    assert any(",ipad" in s for s in names) and not any("concat_views" in s for s in names), names
    # the corners, edges and some of the rest, in 64 bits
    rows = np.r_[0, 1, H - 2, H - 1, rng.integers(2, H - 2, 60)]
    xp = np.pad(x[:, 0].astype(np.float64), ((0, 0), (1, 1), (1, 1)))
    a64, b64, c64 = (v.astype(np.float64) for v in (wa.ravel(), wb, wc.ravel()))
    taps = np.einsum("mckl,c->mkl", b64, a64[5:])  # the 3x3 layer on the single input channel
    for h in rows:
        win = np.stack([xp[:, h + i, j:j + W] for i in range(3) for j in range(3)])  # [9, N, W]
        r64 = np.tensordot(taps.reshape(6, 9), win, axes=1)
        want = (c64[:10] @ a64) * xp[:, h + 1, 1:-1] + np.tensordot(c64[10:], r64, axes=1)
        size = np.abs(c64[:10]) @ np.abs(a64) * np.abs(xp[:, h + 1, 1:-1]) + np.tensordot(
            np.abs(c64[10:]) @ np.abs(np.einsum("mckl,c->mkl", np.abs(b64), np.abs(a64[5:]))).reshape(6, 9), np.abs(win),
            axes=1)
        # 1 + 45 + 16 products summed one after the other
        assert np.all(np.abs(got[:, h] - want) <= 64 * 2.0 ** -24 * size), h
