"""Rows of X gathered on the device in the caller's order, at batches whose
rows leave in one piece and in several (128 MiB each), against the rows of each
structure alone. Equal sums in another order of adds: 1e-12 of a column's
largest entry."""

import numpy as np
import pytest

from pypolymlp_amd import capi, datasets
from pypolymlp_amd.params import ModelSpec

pytestmark = pytest.mark.gpu


# (structures' repetitions, features' precision): one piece; three
# pieces that end among force rows
CASES = {
    "one_piece": ([(2, 2, 2), (3, 2, 2), (2, 2, 3)], capi.PLM_FP64),
    "one_piece_fp32": ([(2, 2, 2), (3, 2, 2), (2, 2, 3)], capi.PLM_MIXED),
    "pieces": ([(7, 7, 7)] * 150 + [(2, 2, 2), (3, 2, 2)], capi.PLM_FP64),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_rows_as_structure_by_structure(name):
    reps, precision = CASES[name]
    spec = ModelSpec(n_type=1, cutoff=4.0, model_type=4, max_p=2, gtinv_order=2, gtinv_maxl=(2,),
                     gaussian_params1=(1.0, 1.0, 1), gaussian_params2=(0.0, 3.0, 4))
    m = capi.Model(spec.as_dict())
    sts = [datasets.config4_structure(seed=k, reps=r) for k, r in enumerate(reps)]

    def batch(ss):
        return capi.Batch(m, [s.axis for s in ss], [s.positions_cartesian for s in ss],
                          [s.types for s in ss])

    X = capi.features_x(m, batch(sts), precision)
    n = [s.positions_cartesian.shape[1] for s in sts]
    off = 7 * len(sts) + 3 * np.concatenate([[0], np.cumsum(n)])
    assert X.shape[0] == off[-1]
    assert (X.nbytes > 2 * 128 * 2**20) == (name == "pieces")
    scale = np.max(np.abs(X), axis=0)
    eps = 1e-12 if precision == capi.PLM_FP64 else 2e-5
    for k, s in enumerate(sts):
        one = capi.features_x(m, batch([s]), precision)
        rows = np.concatenate([[k], len(sts) + 6 * k + np.arange(6), np.arange(off[k], off[k + 1])])
        assert np.all(np.abs(X[rows] - one) <= eps * scale)
