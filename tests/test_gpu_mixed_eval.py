"""Evaluation in the mixed form against 64 bits: energies, forces and stresses of
sets of structures are the FP64 rows of X times the coefficients, to the tolerance
of the FP64 evaluation, through every entry point; a model whose per-atom data
fit the LDS in FP32 only is evaluated in FP32, and plm_eval_noalloc takes the
structures that its 64 MiB hold in the precision asked for."""

import numpy as np
import pytest

from pypolymlp_amd import capi, datasets
from pypolymlp_amd.structure import supercell
from tests.helpers import load_model, poscar
from tests.test_gpu_eval_rows import spec, structure

pytestmark = pytest.mark.gpu

ALLOY = datasets.config2_model()
CASES = {
    "alloy_set": (ALLOY, [(n, (15.0 * n) ** (1 / 3)) for n in (16, 27, 32, 54, 64, 108)] * 2),
    "metal": (spec(max_l=(4,), n_gauss=9), [(n, (18.0 * n) ** (1 / 3)) for n in (1, 9, 54)]),
    "pair": (spec(n_type=2, max_l=(), n_gauss=7), [(n, (9.3 * n) ** (1 / 3)) for n in (8, 64)]),
}


def rows_and_model(sp, sts, precision=capi.PLM_FP64):
    m = capi.Model(sp.as_dict())
    b = capi.Batch(m, [s.axis for s in sts], [s.positions_cartesian for s in sts],
                   [s.types for s in sts])
    X = capi.features_x(m, b, precision)
    scale = np.abs(X).max(axis=0)
    c = np.random.default_rng(1).normal(size=X.shape[1]) / np.where(scale > 1e-8, scale, 1e8)
    m.set_coeffs(c)
    return m, b, X @ c, np.abs(X) @ np.abs(c)


def check(got, sts, y, size, tol):
    E, F, S = got
    n_st, at = len(sts), 7 * len(sts)
    for k, s in enumerate(sts):
        n = 3 * s.n_total
        rows = slice(n_st + 6 * k, n_st + 6 * k + 6)
        assert abs(E[k] - y[k]) <= tol * size[k]
        assert np.abs(S[k] - y[rows]).max() <= tol * size[rows].max() + 1e-2 * tol
        assert np.abs(F[k].reshape(-1) - y[at:at + n]).max() <= tol * size[at:at + n].max() + 1e-2 * tol
        at += n


@pytest.mark.parametrize("name", sorted(CASES))
def test_mixed_evaluation_is_64_bit(name):
    sp, sizes = CASES[name]
    sts = [structure(n, box, sp.n_type, 10 * k + n) for k, (n, box) in enumerate(sizes)]
    m, b, y, size = rows_and_model(sp, sts)
    check(capi.eval_batch(m, b, capi.PLM_MIXED), sts, y, size, 1e-11)
    check(capi.EvalGraph(m, b, capi.PLM_MIXED).run(2), sts, y, size, 1e-11)
    for one in (capi.eval_structure, capi.eval_structure_noalloc):
        e, f, s = zip(*(one(m, t.axis, t.positions_cartesian, t.types, capi.PLM_MIXED) for t in sts))
        check((e, f, s), sts, y, size, 1e-11)


def test_model_past_the_lds_in_fp64():
    """10,648 order parameters a type: 170 KB in FP64, 85 KB in FP32, also where the
    rows of X are built. FP32 sums of up to some thousand terms: 1e-4 of the
    magnitudes."""
    sp = spec(n_type=4, max_l=(10,), n_gauss=21, max_p=1, model_type=3)
    sts = [structure(n, box, 4, n) for n, box in ((2, 4.0), (9, 6.2))]
    m, b, y, size = rows_and_model(sp, sts, capi.PLM_MIXED)
    with pytest.raises(RuntimeError, match="LDS"):
        capi.eval_batch(m, b)
    check(capi.eval_batch(m, b, capi.PLM_MIXED), sts, y, size, 1e-4)


def test_noalloc_limit_counts_the_precision_asked_for():
    sp, coeffs = load_model("polymlp.yaml.gtinv.MgO")
    m = capi.Model(sp.as_dict())
    m.set_coeffs(coeffs)
    st = supercell(poscar("POSCAR.RS.MgO"), [7, 7, 8])  # 3,136 atoms
    args = m, st.axis, st.positions_cartesian, st.types
    with pytest.raises(RuntimeError, match="too large"):
        capi.eval_structure_noalloc(*args)
    got, want = capi.eval_structure_noalloc(*args, capi.PLM_MIXED), capi.eval_structure(*args)
    assert got[0] == pytest.approx(want[0], rel=1e-12)
    assert np.abs(got[1] - want[1]).max() <= 1e-9
