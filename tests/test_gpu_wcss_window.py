"""The wcss fold of training (and with it the convergence test) at the edges of
its chunks (256 terms) and windows (1,024 chunks), on sums that cross binades,
hold ties and outgrow the fp32 range, against the oracle."""
import numpy as np
import pytest

from oracle import binding as orc
from tac_gpu import pq

pytestmark = pytest.mark.gpu
NEVER = float("-inf")


def _check(x, m, ksub, iters=3, tol=NEVER):
    n, dim = x.shape
    init = np.ascontiguousarray(
        x[:ksub].reshape(ksub, m, dim // m).transpose(1, 0, 2))
    got = pq.train(x, dim, 0, m=m, ksub=ksub, max_iters=iters, tol=tol, init_codebooks=init)
    ref = orc.pq_train(x, dim, m, ksub, init=init, max_iters=iters, tol=tol, n_threads=16)
    assert ref.status == 0
    # bit for bit; of a NaN, whose sign and payload IEEE 754 leaves open, that it is one
    nan = np.isnan(ref.wcss)
    assert np.array_equal(np.isnan(got.stats.wcss), nan)
    assert np.array_equal(got.stats.wcss[~nan].view(np.uint32), ref.wcss[~nan].view(np.uint32))
    assert np.array_equal(got.stats.iters_run, ref.iters_run)


@pytest.mark.parametrize("n", [9, 255, 256, 257, 511, 4097, 262_143, 262_144, 262_145, 600_001])
def test_chunk_and_window_edges(gpu, n):
    x = (np.random.default_rng(n).standard_normal((n, 4)) * 0.3).astype(np.float32)
    _check(x, 2, 8)


@pytest.mark.parametrize("kind", ["ties", "growing", "shrinking", "huge", "tiny", "zeros", "nan"])
def test_term_patterns(gpu, kind):
    """ties: integer coordinates; growing / shrinking: a binade every few chunks."""
    n = 20_000
    rng = np.random.default_rng(3)
    x = rng.standard_normal((n, 4)).astype(np.float32)
    ramp = np.exp2(np.linspace(-30, 30, n)).astype(np.float32)[:, None]
    if kind == "ties":
        x = rng.integers(-40, 40, (n, 4)).astype(np.float32)
    elif kind == "growing":
        x *= ramp
    elif kind == "shrinking":
        x *= ramp[::-1]
    elif kind == "huge":
        x *= np.float32(1e18)
    elif kind == "tiny":
        x *= np.float32(1e-21)
    elif kind == "zeros":
        x[100:] = x[rng.integers(0, 8, n - 100)]
    else:
        x[7000, 1] = np.nan
    _check(x, 2, 8)


def test_convergence_is_the_oracles(gpu):
    x = (np.random.default_rng(8).standard_normal((50_000, 16)) * 0.3).astype(np.float32)
    _check(x, 4, 64, iters=25, tol=1e-3)


@pytest.mark.parametrize("n", [1_521_797, 8_000_000])
def test_sum_a_binade_behind(gpu, n):
    """Equal terms: the serial fp32 sum falls behind the f64 prefix that places
    the chunks' candidate binades (88 chunks of 1,521,797 terms, 439 of 8,000,000)."""
    x = np.full((n, 1), 0.7, np.float32)
    x[::2] *= -1
    init = np.zeros((1, 1, 1), np.float32)
    got = pq.train(x, 1, 0, m=1, ksub=1, max_iters=1, tol=NEVER, init_codebooks=init)
    ref = orc.pq_train(x, 1, 1, 1, init=init, max_iters=1, tol=NEVER, n_threads=1)
    assert ref.status == 0
    assert np.array_equal(got.stats.wcss.view(np.uint32), ref.wcss.view(np.uint32))
