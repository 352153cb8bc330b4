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
