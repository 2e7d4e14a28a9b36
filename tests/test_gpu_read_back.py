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


def test_model_without_features():
    """No radial function in any type pair: rows are refused, as their kernels
    have nothing to launch, and the normal equations are empty."""
    spec = ModelSpec(n_type=1, cutoff=4.0, feature_type="pair", model_type=2, max_p=2,
                     gtinv_order=0, gtinv_maxl=(), gaussian_params1=(1.0, 1.0, 1),
                     gaussian_params2=(0.0, 3.0, 4), pair_params_conditional={(0, 0): []})
    m = capi.Model(spec.as_dict())
    assert m.n_features == 0
    s = datasets.config4_structure(reps=(2, 2, 2))
    b = capi.Batch(m, [s.axis], [s.positions_cartesian], [s.types])
    with pytest.raises(RuntimeError):
        capi.features_x(m, b)
    xtx, xty, s1, s2, y_sq, n = capi.Normal(m).result()
    assert xtx.shape == (0, 0) and xty.shape == (0,) and y_sq == 0.0 and n == 0
