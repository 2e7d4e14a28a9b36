"""The device memory pool: buffers handed on between calls of other sizes,
models and threads leave every result as it was. Repeated FP64 evaluations
differ by the order of atomic sums only (2e-13 of the largest value allows for
about 1e3 rounding errors)."""

import threading

import numpy as np
import pytest

from pypolymlp_amd import capi, datasets, mlp_dev

pytestmark = pytest.mark.gpu


def close(a, b):
    return np.abs(a - b).max() <= 2e-13 * np.abs(b).max()


def job(spec, structures, seed):
    """A model with random coefficients and its evaluations and X rows."""
    m = capi.Model(spec.as_dict())
    m.set_coeffs(np.random.default_rng(seed).normal(size=m.n_features))

    def run():
        b = capi.Batch(m, [s.axis for s in structures],
                       [s.positions_cartesian for s in structures], [s.types for s in structures])
        e, f, s = capi.eval_batch(m, b)
        return np.concatenate([e, np.concatenate(f).ravel(), s.ravel()]), capi.features_x(m, b)

    return run


def test_results_across_sizes_and_threads():
    sts = datasets.config2_dataset(7, targets=False).structures
    metal = [datasets.config4_structure(reps=(4, 4, 3 + k)) for k in range(3)]
    jobs = [job(datasets.config1_model(), metal[:1], 1), job(datasets.config1_model(), metal, 2),
            job(datasets.config2_model(), sts[:2], 3), job(datasets.config2_model(), sts, 4)]
    first = [j() for j in jobs]
    again = [j() for j in reversed(jobs)][::-1]
    for (a, x), (b, y) in zip(again, first):
        assert close(a, b) and close(x, y)
    out = [None] * len(jobs)

    def work(k):
        out[k] = [jobs[k]() for _ in range(6)]

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(jobs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for got, (b, y) in zip(out, first):
        for a, x in got:
            assert close(a, b) and close(x, y)


def test_ridge_after_larger_buffers():
    """A small system solved in recycled buffers of larger ones."""
    res = []
    for F in (700, 130, 700, 65, 130):
        A = np.random.default_rng(F).normal(size=(2 * F, F))
        A = A.T @ A
        c = mlp_dev.solver_ridge(A, A @ np.ones(F), np.array([1e-9, 1e-8]))
        res.append(np.abs(c - 1.0).max())
    assert max(res) < 1e-6


def test_idle_memory_is_given_back_on_request():
    """A model keeps the pool's idle blocks alive (a GiB and more of X here);
    they are free for another allocator after release_memory, and results stay."""
    import torch

    spec = datasets.config1_model()
    sts = [datasets.config4_structure(seed=k, reps=(4, 4, 4)) for k in range(120)]
    run = job(spec, sts, 5)
    first = run()
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    given = capi.release_memory()
    assert given >= 1 << 30
    assert torch.cuda.mem_get_info()[0] - free >= given // 2
    assert capi.release_memory() == 0
    for a, b in zip(run(), first):
        assert close(a, b)
