"""A batch is complete when its creation returns: no device work is left that a
later call would wait for, or report the failure of."""

import time

import numpy as np
import pytest
import torch

from pypolymlp_amd import capi, datasets

pytestmark = pytest.mark.gpu


def test_no_work_is_left_after_creation():
    """400 cells of 1,000 atoms by the search over all pairs, whose fill takes
    about 4 ms; waiting for an idle device takes some microseconds."""
    m = capi.Model(datasets.config1_model().as_dict())
    rng = np.random.default_rng(2)
    axes = [np.diag([26.0, 26.0, 26.0])] * 400
    pos = [np.ascontiguousarray(26.0 * rng.uniform(size=(3, 1000))) for _ in axes]
    types = [np.zeros(1000, dtype=int)] * 400
    capi.Batch(m, axes[:1], pos[:1], types[:1])
    torch.cuda.synchronize()
    b = capi.Batch(m, axes, pos, types)
    t = time.perf_counter()
    torch.cuda.synchronize()
    assert time.perf_counter() - t < 2e-3
    assert b.n_pairs > 0
