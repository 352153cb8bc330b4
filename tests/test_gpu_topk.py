"""TopK's replay of the reference heap as a pipeline of insertions: rows whose
values tie across the k-th place, at heap depths 1 to 11, against the oracle."""

from __future__ import annotations

import numpy as np
import pytest

from spinnv2_amd.spk import models, write_spk

from .helpers import run_gpu, run_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("largest", [0, 1])
@pytest.mark.parametrize("dim,k", [(2, 1), (5, 2), (9, 3), (70, 4), (65, 64), (400, 127), (3000, 128), (1025, 1024),
                                   (16384, 1023), (16385, 1024)])
def test_topk_tied_rows(gpu, dim, k, largest):
    rng = np.random.default_rng(dim + k)
    x = np.stack([np.round(rng.standard_normal(dim) * 4),           # many ties, few insertions
                  np.sort(np.round(rng.standard_normal(dim) * 50)),  # every element enters (largest) ...
                  np.sort(np.round(rng.standard_normal(dim) * 50))[::-1],  # ... or none
                  np.round(rng.standard_normal(dim) * 1000) / 8]).astype(np.float32)
    x[3, -1] = x[3, 0]
    g = models.index_op("TopK", [4, dim], k=k, axis=1, largest=largest)
    blob = write_spk(g, "mi355x")
    got, want = run_gpu(blob, [x], 2), run_oracle(blob, [x])
    np.testing.assert_array_equal(got[0].view(np.uint32), want[0].view(np.uint32))
    np.testing.assert_array_equal(got[1], want[1])
