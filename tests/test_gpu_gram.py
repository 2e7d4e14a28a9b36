"""FP64 normal equations at the edges of the Gram's tiles (128 columns), of its
row splits (512 rows each) and of its whole rounds (512 tiles), against the
product of the rows that plm_features_x gives. A sum of n products is within
n eps of the product of the columns' norms, whatever its order."""

import numpy as np
import pytest

from pypolymlp_amd import capi, datasets
from pypolymlp_amd.params import ModelSpec

pytestmark = pytest.mark.gpu


def model(n_gauss, max_l, max_p=2, n_type=1, model_type=4):
    return ModelSpec(n_type=n_type, cutoff=5.0, model_type=model_type, max_p=max_p,
                     gtinv_order=len(max_l) + 1, gtinv_maxl=max_l,
                     gaussian_params1=(1.0, 1.0, 1), gaussian_params2=(0.0, 4.0, n_gauss))


# (model, structures): 1 tile and few rows; one column short of and past whole
# tiles with [X | y]; row splits down to 512 rows; more than 512 tiles (4,395
# columns: 630) with one round in whole rows and the rest in three row splits, the
# last of them shorter (1,856 padded rows: 624, 624 and 608)
CASES = {
    "one_tile": (model(2, (2,)), 1),
    "two_tiles": (model(4, (2,)), 7),
    "split_512": (model(7, (4,)), 7),
    "split_many": (model(6, (4,)), 60),
    "many_tiles": (model(14, (4, 4)), 13),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_fp64_gram(name):
    spec, n_st = CASES[name]
    rng = np.random.default_rng(n_st)
    sts = [datasets.config4_structure(seed=k, reps=(3, 3, 2 + k % 2)) for k in range(n_st)]
    m = capi.Model(spec.as_dict())
    b = capi.Batch(m, [s.axis for s in sts], [s.positions_cartesian for s in sts],
                   [s.types for s in sts])
    X = capi.features_x(m, b)
    n, F = X.shape
    w, y = rng.uniform(0.1, 1.0, size=n), rng.normal(size=n)
    acc = capi.Normal(m)
    for _ in range(2):  # the second pass adds to sums that are there
        acc.accumulate(b, w, y)
    xtx, xty, _, _, y_sq, _ = acc.result()
    A = np.concatenate([X * w[:, None], y[:, None]], axis=1)
    G = 2.0 * (A.T @ A)
    norm = np.sqrt(np.diag(G))
    got = np.zeros_like(G)
    got[:F, :F], got[:F, F], got[F, :F], got[F, F] = xtx, xty, xty, y_sq
    # the rows are rebuilt with another order of atomic sums: 1e-14 of the entries
    tol = (4.0 * n * np.finfo(float).eps + 1e-13) * np.outer(norm, norm)
    print(name, F, n, float(np.max(np.abs(got - G) / tol)))
    assert np.all(np.abs(got - G) <= tol)
