"""k-means++ seeding at the edges of its runs (512 rows), blocks (4,096) and of
the rows whose blocks draw for themselves (262,144), against the oracle."""
import numpy as np
import pytest

from oracle import binding as orc
from tac_gpu import errors, pq

pytestmark = pytest.mark.gpu
NEVER = float("-inf")


def _rows(n, dim, seed, distinct=None):
    rng = np.random.default_rng(seed)
    x = (rng.standard_normal((distinct or n, dim)) * 0.3).astype(np.float32)
    return x[rng.integers(0, distinct, n)] if distinct else x


@pytest.mark.parametrize("n,m,dsub,ksub", [(20, 4, 2, 16), (512, 2, 4, 40), (513, 3, 3, 40),
                                           (4096, 2, 8, 64), (4097, 32, 2, 100), (40_000, 1, 1, 1000),
                                           (262_144, 2, 4, 32), (262_145, 2, 4, 32),
                                           (300_001, 3, 8, 20)])
@pytest.mark.parametrize("exact", [False, True])
def test_seeds_match_oracle(gpu, monkeypatch, n, m, dsub, ksub, exact):
    # One Lloyd iteration from the seeds: any other pick changes its means.
    if exact and ksub > 100:
        ksub = 60
    x = _rows(n, m * dsub, n + m, distinct=n // 3 if n % 2 else None)
    if exact:
        monkeypatch.setenv("TAC_GPU_KPP_EXACT", "1")
    got = pq.train(x, m * dsub, 77, m=m, ksub=ksub, max_iters=1, tol=NEVER)
    ref = orc.pq_train(x, m * dsub, m, ksub, seed=77, max_iters=1, tol=NEVER, n_threads=16)
    assert ref.status == 0
    assert np.array_equal(got.codebooks.view(np.uint32), ref.codebooks.reshape(-1).view(np.uint32))


@pytest.mark.parametrize("n,m,dsub,ksub", [(5000, 8, 4, 100), (513, 3, 2, 150), (100_001, 5, 8, 70),
                                           (270_001, 3, 4, 40)])
@pytest.mark.parametrize("every", [2, 3, 7, 40])
def test_open_draws_between_decided_ones(gpu, monkeypatch, n, m, dsub, ksub, every):
    """Only some draws of some subspaces are left open: the drawn run's weights
    go back from the patch, the exact draw resumes the subspace, and it catches
    up while the others pass by (every 32 rounds, and at the end).  The 513 rows
    hold some 221 distinct ones: more seeds than that would be AllZero."""
    x = _rows(n, m * dsub, n + every, distinct=n // 2 if n % 2 else None)
    monkeypatch.setenv("TAC_GPU_KPP_EXACT", str(every))
    got = pq.train(x, m * dsub, 77, m=m, ksub=ksub, max_iters=1, tol=NEVER)
    ref = orc.pq_train(x, m * dsub, m, ksub, seed=77, max_iters=1, tol=NEVER, n_threads=16)
    assert ref.status == 0
    assert np.array_equal(got.codebooks.view(np.uint32), ref.codebooks.reshape(-1).view(np.uint32))


@pytest.mark.parametrize("n", [3000, 270_000])
def test_errors_of_the_lowest_subspace(gpu, n):
    """All weights zero after the first pick, and distances that overflow."""
    x = _rows(n, 8, 3)
    x[:, 4:] = 0.25
    with pytest.raises(errors.AllZero):
        pq.train(x, 8, 1, m=2, ksub=8, max_iters=1, tol=NEVER)
    x[:, 2] = np.where(np.arange(n) % 2, 3e38, -3e38)
    with pytest.raises(errors.NonFinite):
        pq.train(x, 8, 1, m=2, ksub=8, max_iters=1, tol=NEVER)
    got = pq.train(_rows(n, 8, 4), 8, 1, m=2, ksub=8, max_iters=1, tol=NEVER)
    ref = orc.pq_train(_rows(n, 8, 4), 8, 2, 8, seed=1, max_iters=1, tol=NEVER, n_threads=16)
    assert np.array_equal(got.codebooks.view(np.uint32), ref.codebooks.reshape(-1).view(np.uint32))
