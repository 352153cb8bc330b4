"""SPKV2_TUNE_DB: a later process reuses the measured tile choices, hybrid
schedules included (their split is stored as 1000 + slices per remaining
tile)."""

from __future__ import annotations

import json
import os
import subprocess
import sys
from pathlib import Path

import numpy as np
import pytest

from .helpers import rng_inputs

pytestmark = pytest.mark.gpu

ROOT = Path(__file__).resolve().parents[1]

# one conv with enough tiles for the hybrid schedule; prints its kernel name
# and a checksum of its output
CHILD = r"""
import json, sys
sys.path.insert(0, %r)
import numpy as np
from spinnv2_amd.runtime import Model
from spinnv2_amd.spk import models, write_spk
g = models.single_conv(4, 16, 63, 67, 200, 3, 1, 1, act="Relu")
x = models.make_input(g.tensors[g.inputs[0]].shape, 11)
with Model(write_spk(g, "mi355x")) as m:
    m.set_input(0, x)
    m.run()
    y = m.get_output(0)
    print(json.dumps({"name": m.kernel_name(0), "sum": float(np.abs(y).sum())}))
""" % str(ROOT)


def _child(db: Path) -> dict:
    env = dict(os.environ, SPKV2_TUNE_DB=str(db))
    for k in ("SPKV2_CONV_CFG", "SPKV2_CONV_SPLITK", "SPKV2_CONV_HYBRID", "SPKV2_CONV_TUNE"):
        env.pop(k, None)
    out = subprocess.run([sys.executable, "-c", CHILD], env=env, capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr[-2000:]
    return json.loads(out.stdout.strip().splitlines()[-1])


NETWORK_CHILD = r"""
import hashlib, json, sys
sys.path.insert(0, %r)
from spinnv2_amd.runtime import Model
from spinnv2_amd.spk import models, write_spk
g = models.resnet(101, 1)
x = models.make_input(g.tensors[g.inputs[0]].shape, 5)
with Model(write_spk(g, "mi355x")) as m:
    m.set_input(0, x)
    m.run()
    y = m.get_output(0)
    names = [m.kernel_name(n.id) for n in g.nodes if n.op_type in ("Conv", "Gemm")]
print(json.dumps({"sha": hashlib.sha256(y.tobytes()).hexdigest(), "names": names}))
""" % str(ROOT)


def test_benchmark_network_is_bit_reproducible_across_processes(gpu):
    """The committed tune table (spinnv2_amd/lib/mi355x.tune) fixes the tile
    and split-K choice of every ResNet-101 layer, so two fresh processes
    without a tune DB of their own pick the same kernels and produce the
    same logits bit for bit."""
    assert (ROOT / "spinnv2_amd" / "lib" / "mi355x.tune").stat().st_size > 0
    env = dict(os.environ)
    for k in ("SPKV2_TUNE_DB", "SPKV2_TUNE_TABLE", "SPKV2_CONV_CFG", "SPKV2_CONV_SPLITK", "SPKV2_CONV_HYBRID",
              "SPKV2_CONV_TUNE"):
        env.pop(k, None)
    runs = []
    for _ in range(2):
        out = subprocess.run([sys.executable, "-c", NETWORK_CHILD], env=env, capture_output=True, text=True,
                             timeout=100)
        assert out.returncode == 0, out.stderr[-2000:]
        runs.append(json.loads(out.stdout.strip().splitlines()[-1]))
    assert runs[0]["names"] == runs[1]["names"]
    assert runs[0]["sha"] == runs[1]["sha"]


def test_tune_db_reuses_hybrid_choice(gpu, tmp_path):
    db = tmp_path / "tune.db"
    first = _child(db)
    lines = db.read_text().split("\n")
    conv = [ln for ln in lines if ln.startswith("conv|")]
    assert len(conv) == 1, lines
    key, cfg, _ = conv[0].split()
    # replace the measured choice with a hybrid schedule of 4 slices
    db.write_text(f"{key} {cfg} 1004\n")
    second = _child(db)
    assert ",dp=" in second["name"], second
    assert abs(second["sum"] - first["sum"]) <= 1e-4 * first["sum"]
    assert db.read_text() == f"{key} {cfg} 1004\n"  # a hit stores nothing new


# entries of conv_f32.hip's tile table that run the implicit-GEMM kernel
# (64- and 128-row tiles, BK 16 to 128, the 32- and 96-row tiles); the
# skinny (12, 13) and thin (17, 18) kernels sum in orders of their own
IGEMM_CFGS = [0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 14, 15, 16, 19, 20, 25, 26]


def test_igemm_tiles_share_one_summation_order(gpu, monkeypatch):
    """The deterministic tuner's premise: every implicit-GEMM tile shape
    gives the same fp32 bits for the same split-K cut (k = 1024: one slice,
    or four slices of 256 k, as 16 k-tiles of 16, 8 of 32 or 4 of 64), so
    timing may choose among them freely."""
    from spinnv2_amd.runtime import Model
    from spinnv2_amd.spk import models, write_spk

    from .helpers import rng_inputs

    g = models.single_conv(2, 1024, 14, 14, 96, 1, act=None, residual=True)
    blob = write_spk(g, "mi355x")
    xs = rng_inputs(g)
    monkeypatch.setenv("SPKV2_CONV_TUNE", "0")
    for split, cfgs in ((1, IGEMM_CFGS), (4, [6, 7, 8])):
        outs = []
        for c in cfgs:
            monkeypatch.setenv("SPKV2_CONV_CFG", str(c))
            monkeypatch.setenv("SPKV2_CONV_SPLITK", str(split))
            with Model(blob) as m:
                for i, x in enumerate(xs):
                    m.set_input(i, x)
                m.run()
                outs.append((m.kernel_name(0), m.get_output(0)))
        names = [n for n, _ in outs]
        assert len(set(names)) == len(cfgs) and all(f"splitk={split}>" in n for n in names), names
        for n, y in outs[1:]:
            np.testing.assert_array_equal(y.view(np.uint32), outs[0][1].view(np.uint32), err_msg=f"{n} vs {names[0]}")


DET_CHILD = r"""
import hashlib, json, sys
sys.path.insert(0, %r)
from spinnv2_amd.runtime import Model
from spinnv2_amd.spk import models, write_spk
g = models.resnet(18, 3, image=72)
x = models.make_input(g.tensors[g.inputs[0]].shape, 9)
with Model(write_spk(g, "mi355x")) as m:
    m.set_input(0, x)
    m.run()
    y = m.get_output(0)
    names = [m.kernel_name(n.id) for n in g.nodes if n.op_type in ("Conv", "Gemm")]
print(json.dumps({"sha": hashlib.sha256(y.tobytes()).hexdigest(), "names": names}))
""" % str(ROOT)


def test_deterministic_tuner_is_bit_reproducible_outside_the_table(gpu):
    """SPKV2_TUNE_DETERMINISTIC=1 on layer shapes the committed table does
    not hold (ResNet-18 at 72x72, batch 3), tuned live in two fresh
    processes with different tie bands (0% and 50%: different tile picks
    within a summation order): the model fixes each layer's summation order,
    so the logits are bit-identical whatever the timings."""
    runs = []
    for tie in ("0", "50"):
        env = dict(os.environ, SPKV2_TUNE_TABLE="0", SPKV2_TUNE_TIE=tie, SPKV2_TUNE_DETERMINISTIC="1")
        for k in ("SPKV2_TUNE_DB", "SPKV2_CONV_CFG", "SPKV2_CONV_SPLITK", "SPKV2_CONV_HYBRID", "SPKV2_CONV_TUNE"):
            env.pop(k, None)
        out = subprocess.run([sys.executable, "-c", DET_CHILD], env=env, capture_output=True, text=True, timeout=100)
        assert out.returncode == 0, out.stderr[-2000:]
        runs.append(json.loads(out.stdout.strip().splitlines()[-1]))
    print("tile picks that differ:", [(a, b) for a, b in zip(runs[0]["names"], runs[1]["names"]) if a != b])
    assert runs[0]["sha"] == runs[1]["sha"]


def test_tuner_times_ordinary_operands(gpu, monkeypatch, capfd):
    """The tuner's time of its choice is that of ordinary values (at which
    the chip lowers its clock: 20% here), not that of zeros, which is below
    the layer's node time on zeros by what the node's events take."""
    from spinnv2_amd.runtime import Model
    from spinnv2_amd.spk import models, write_spk

    for k in ("SPKV2_TUNE_DB", "SPKV2_CONV_CFG", "SPKV2_CONV_SPLITK", "SPKV2_CONV_HYBRID", "SPKV2_CONV_TUNE"):
        monkeypatch.delenv(k, raising=False)
    monkeypatch.setenv("SPKV2_TUNE_LOG", "1")
    monkeypatch.setenv("SPKV2_TUNE_TIE", "0")  # the fastest candidate, first in the log
    took = {}
    for name in ("ordinary", "zeros"):
        g = models.single_conv(48, 272, 29, 29, 256, 3, act=None)
        x = np.random.default_rng(1).standard_normal((48, 272, 29, 29)).astype(np.float32)
        if name == "zeros":
            x[:] = 0
            g.tensors[g.nodes[0].inputs[1]].data[:] = 0
        with Model(write_spk(g, "mi355x")) as mdl:
            mdl.set_profiling(True)
            mdl.set_input(0, x)
            for _ in range(10):
                mdl.run()
            mdl.reset_node_times()
            for _ in range(30):
                mdl.run()
            ms, runs = mdl.node_time(0)[:2]
            took[name] = 1e3 * ms / runs
    tuned = [line for line in capfd.readouterr().err.splitlines() if line.startswith("[tune]   ")]
    best = float(tuned[0].split()[-1])
    assert best > took["zeros"], (best, took)


def test_tuner_times_the_padding_that_runs(gpu, monkeypatch, capfd):
    """A padded layer that pads its own input is tuned with its copy or its
    checked taps, as it runs then; one whose input another layer hands over
    padded is tuned on padded planes."""
    from spinnv2_amd.runtime import Model
    from spinnv2_amd.spk import models, write_spk
    from spinnv2_amd.spk.graph import Graph

    for k in ("SPKV2_TUNE_DB", "SPKV2_CONV_CFG", "SPKV2_CONV_SPLITK", "SPKV2_CONV_HYBRID", "SPKV2_CONV_TUNE",
              "SPKV2_IMPLICIT_PAD"):
        monkeypatch.delenv(k, raising=False)
    monkeypatch.setenv("SPKV2_TUNE_LOG", "1")
    monkeypatch.setenv("SPKV2_TUNE_TIE", "0")  # the fastest candidate, first in the log

    def tuned(g):
        """Per layer the log's candidates, and the kernel that runs."""
        capfd.readouterr()
        with Model(write_spk(g, "mi355x")) as mdl:
            mdl(*rng_inputs(g))
            names = [mdl.kernel_name(i) for i in range(len(g.nodes))]
        layers = []
        for line in capfd.readouterr().err.splitlines():
            if line.startswith("[tune] conv"):
                layers.append([])
            elif line.startswith("[tune]   ") and layers:
                layers[-1].append(line)
        return layers, names

    forms = set()
    for n, c, h, w, m, s in [(4, 40, 23, 19, 72, 1), (6, 104, 35, 27, 72, 2), (2, 10, 61, 53, 40, 1)]:
        (lines,), (name,) = tuned(models.single_conv(n, c, h, w, m, 3, s, 1))
        for line in lines:
            assert (",copy" in line) != (",ipad" in line), line
            forms.add(",ipad" if ",ipad" in line else ",copy")
        assert (",ipad" in lines[0]) == (",ipad" in name), (lines[0], name)
    assert len(forms) == 2, forms

    g = Graph("two")
    rng = np.random.default_rng(5)
    y = g.input("x", [3, 40, 21, 19])
    for k, pad in ((1, 0), (3, 1)):
        y = g.conv(y, rng.standard_normal((40, 40, k, k)).astype(np.float32), np.zeros(40, np.float32), pad=pad)
    g.mark_output(y)
    layers, names = tuned(g)
    assert "+handoff" in names[1], names
    assert len(layers) == 2 and not any(",copy" in line or ",ipad" in line for lines in layers for line in lines)
