"""Evaluation against the rows of X: for coefficients c the energies, forces and
stresses are the energy, force and stress rows times c, and the rows come from
kernels of their own. FP64, 1e-11 of the largest value per structure (sums of
up to some thousand terms); at radial functions that do not fill the pair loop's
rows of four, at each of its bounds on max_l, with neighbours around and past
the 64 of an order-parameter chunk and more tiles than that form holds, with
few pairs (keys split over workgroups), with type pairs of unequal and no radial
functions. Cells of many atoms and pairs (a wave per atom in the contraction,
unsplit keys, energies and stresses summed by several workgroups) are periodic
replicas of a small cell whose rows are known."""

import numpy as np
import pytest

from pypolymlp_amd import capi
from pypolymlp_amd.params import ModelSpec
from pypolymlp_amd.structure import PolymlpStructure

pytestmark = pytest.mark.gpu


def structure(n, box, n_type, seed):
    rng = np.random.default_rng(seed)
    side = int(np.ceil(n ** (1 / 3)))
    grid = np.mgrid[0:side, 0:side, 0:side].reshape(3, -1)[:, :n] / side
    axis = np.diag(np.full(3, box)) + rng.normal(0, 0.05, (3, 3))
    frac = grid + rng.normal(0, 0.02, grid.shape)
    types = rng.integers(0, n_type, size=n)
    return PolymlpStructure(axis=axis, positions=frac, types=[int(t) for t in types],
                            n_atoms=[int(np.sum(types == t)) for t in range(n_type)],
                            elements=[chr(65 + t) for t in types])


def spec(n_type=1, max_l=(4,), n_gauss=4, max_p=2, model_type=4, cond=None, **kw):
    return ModelSpec(n_type=n_type, cutoff=5.0, feature_type="gtinv" if max_l else "pair",
                     model_type=model_type if max_l else 2, max_p=max_p,
                     gtinv_order=len(max_l) + 1, gtinv_maxl=max_l,
                     gaussian_params1=(1.0, 1.0, 1), gaussian_params2=(0.0, 4.0, n_gauss),
                     pair_params_conditional=cond, **kw)


SMALL = [(1, 3.1), (2, 4.0), (9, 6.2)]
LARGE = SMALL + [(64, 11.0), (200, 17.0)]
MANY = [(1500, 32.0)]
DENSE = [(8, 4.2), (27, 6.0), (64, 6.5), (125, 9.0)]  # 55, 65, 120, 90 neighbours
COND = {(0, 0): [0, 1, 2, 3, 4], (0, 1): [0, 2, 3], (1, 1): [1]}
NONE = {(0, 0): [0, 1, 2], (0, 1): [], (1, 1): [0, 1, 2, 4]}

CASES = {
    "l1": (spec(max_l=(1,), n_gauss=1), SMALL),
    "l3_n4": (spec(max_l=(3,), n_gauss=3), LARGE),
    "l4_n5": (spec(max_l=(4,), n_gauss=4), LARGE),
    "l4_many": (spec(max_l=(4,), n_gauss=7), MANY),
    "l5": (spec(max_l=(5, 3), n_gauss=2, model_type=3), SMALL),
    "l8_n9": (spec(max_l=(8,), n_gauss=8, n_type=2, model_type=3), LARGE),
    "l9": (spec(max_l=(9,), n_gauss=3), SMALL),
    "l12_n17": (spec(max_l=(12,), n_gauss=16, model_type=3), SMALL),
    "cond": (spec(n_type=2, max_l=(4, 2), model_type=3, cond=COND), LARGE),
    "cond_none": (spec(n_type=2, max_l=(2,), cond=NONE), LARGE),
    "dense": (spec(max_l=(4,), n_gauss=6), DENSE),
    "dense_alloy": (spec(n_type=3, max_l=(6,), n_gauss=3, model_type=3), DENSE),
    "dense_pair": (spec(n_type=2, max_l=(), n_gauss=5), DENSE),
    "tiles_beyond": (spec(n_type=4, max_l=(10,), n_gauss=19, max_p=1, model_type=3), SMALL),
    "order3_p3": (spec(n_type=3, max_l=(4, 2), n_gauss=1, max_p=3, model_type=3), SMALL),
    "pair": (spec(n_type=2, max_l=(), n_gauss=6), LARGE),
    "pair_many": (spec(n_type=2, max_l=(), n_gauss=5, cond=COND), MANY),
}


@pytest.mark.parametrize("form", ["", "records"])
@pytest.mark.parametrize("name", sorted(CASES))
def test_eval_matches_rows(name, form, monkeypatch):
    if form:
        monkeypatch.setenv("PLM_EVAL_PAIR", form)
    sp, sizes = CASES[name]
    sts = [structure(n, box, sp.n_type, n) for n, box in sizes]
    m = capi.Model(sp.as_dict())
    b = capi.Batch(m, [s.axis for s in sts], [s.positions_cartesian for s in sts],
                   [s.types for s in sts])
    X = capi.features_x(m, b)
    scale = np.abs(X).max(axis=0)
    c = np.random.default_rng(1).normal(size=X.shape[1]) / np.where(scale > 1e-8, scale, 1e8)
    m.set_coeffs(c)
    E, F, S = capi.eval_batch(m, b)
    y, n_st = X @ c, len(sts)
    size = np.abs(X) @ np.abs(c)
    at = 7 * n_st
    for k, s in enumerate(sts):
        n = 3 * s.n_total
        assert abs(E[k] - y[k]) <= 1e-11 * size[k]
        rows = slice(n_st + 6 * k, n_st + 6 * k + 6)
        assert np.abs(S[k] - y[rows]).max() <= 1e-11 * size[rows].max() + 1e-13
        assert np.abs(F[k].reshape(-1) - y[at:at + n]).max() <= 1e-11 * size[at:at + n].max() + 1e-13
        at += n


# from 8,192 atoms on a wave per atom contracts, from 2,048 waves of half pairs on
# a lane takes all keys, from 4,096 on several workgroups add a structure up
REPLICAS = {
    "metal": (spec(max_l=(2,), n_gauss=3), 7),
    "pair": (spec(n_type=2, max_l=(), n_gauss=5), 7),
    "alloy": (spec(n_type=2, max_l=(4, 2), n_gauss=3, model_type=3), 6),
}


@pytest.mark.parametrize("precision", [capi.PLM_FP64, capi.PLM_MIXED])
@pytest.mark.parametrize("name", sorted(REPLICAS))
def test_large_cell_matches_rows_of_its_unit(name, precision):
    sp, reps = REPLICAS[name]
    s = structure(54, 9.3, sp.n_type, 3)
    pos, types = s.positions_cartesian, np.array(s.types)
    m = capi.Model(sp.as_dict())
    b = capi.Batch(m, [s.axis], [pos], [types])
    X = capi.features_x(m, b)
    scale = np.abs(X).max(axis=0)
    c = np.random.default_rng(1).normal(size=X.shape[1]) / np.where(scale > 1e-8, scale, 1e8)
    m.set_coeffs(c)
    y, size = X @ c, np.abs(X) @ np.abs(c)
    cells = np.mgrid[0:reps, 0:reps, 0:reps].reshape(3, -1)
    n = cells.shape[1]
    large = (pos[:, None, :] + (s.axis @ cells)[:, :, None]).reshape(3, -1)
    big = capi.Batch(m, [s.axis * reps], [large], [np.tile(types, n)])
    assert 54 * n >= 8192 and big.n_pairs // 2 >= 64 * (4096 if name != "alloy" else 2048)
    E, F, S = capi.eval_batch(m, big, precision)
    assert abs(E[0] - n * y[0]) <= 1e-11 * n * size[0]
    assert np.abs(S[0] - n * y[1:7]).max() <= 1e-11 * n * size[1:7].max()
    assert np.abs(F[0].reshape(n, -1) - y[7:]).max() <= 1e-11 * size[7:].max()


@pytest.mark.parametrize("max_p,model_type", [(2, 4), (3, 3)])
def test_fp32_energy_rows(max_p, model_type):
    """Energy rows with 16 atoms' factors in flight: atom counts around that,
    two and three factors. FP32 features within 1e-5 of the sum
    of their magnitudes (some 1e-6 per factor, three factors)."""
    sp = spec(max_l=(2,), n_gauss=3, max_p=max_p, model_type=model_type)
    sts = [structure(n, 3.1 * n ** (1 / 3), 1, n) for n in (1, 3, 4, 5, 15, 16, 17, 33, 64, 65)]
    m = capi.Model(sp.as_dict())
    b = capi.Batch(m, [s.axis for s in sts], [s.positions_cartesian for s in sts],
                   [s.types for s in sts])
    x64 = capi.features_x(m, b)[:len(sts)]
    x32 = capi.features_x(m, b, capi.PLM_MIXED)[:len(sts)]
    per_atom = np.abs(x64) / np.array([s.n_total for s in sts])[:, None]
    size = per_atom.max(axis=0) * np.array([s.n_total for s in sts])[:, None]
    assert np.all(np.abs(x32 - x64) <= 1e-5 * size)
