"""PQ.encode of few rows (encode_small_kernel) at the edges of its rows per
block (16 and 64), its lane widths and its range, against the oracle."""
import numpy as np
import pytest

from oracle import binding as orc
from tac_gpu import device, errors, lib, pq

pytestmark = pytest.mark.gpu


def _encode(x, cb, m, ksub):
    n, dim = x.shape
    got = pq.PQ(dim, dim // m, cb.reshape(-1), m, ksub).encode_many(x)
    dx, dcb = device.DeviceArray.from_host(x), device.DeviceArray.from_host(cb)
    dc = device.DeviceArray((n, m), pq.code_dtype(ksub))
    errors.check(lib.tac_pq_encode_device_noalloc(dx.ptr, n, dim, m, ksub, dcb.ptr, dc.ptr, None))
    device.synchronize()
    assert np.array_equal(dc.to_host(), got)
    return got


@pytest.mark.parametrize("dsub,m,ksub", [(1, 64, 256), (2, 32, 256), (3, 21, 64), (4, 16, 256),
                                         (4, 16, 1024), (4, 5, 1), (5, 4, 3), (6, 5, 31), (7, 3, 17),
                                         (8, 16, 256), (8, 2, 1000)])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 1000, 8192, 8193, 16_383, 16_384])
def test_rows_and_lane_widths(gpu, dsub, m, ksub, n):
    rng = np.random.default_rng(dsub * 1000 + ksub + n)
    x = (rng.standard_normal((n, m * dsub)) * 0.2).astype(np.float32)
    cb = (rng.standard_normal((m, ksub, dsub)) * 0.2).astype(np.float32)
    cb[:, ksub // 2:] = cb[:, :ksub - ksub // 2]  # exact ties: the lowest index wins
    want = orc.pq_encode(x, m * dsub, m, ksub, cb, n_threads=8)
    assert np.array_equal(_encode(x, cb, m, ksub), want)


@pytest.mark.parametrize("dsub,m,ksub,n,small", [
    (1, 256, 64, 12_288, True), (1, 256, 64, 12_289, False), (2, 192, 64, 9557, True),
    (2, 192, 64, 9558, False), (3, 81, 1024, 16_181, True), (3, 81, 1024, 16_182, False),
    (4, 128, 256, 8192, True), (4, 128, 256, 8193, False), (8, 96, 256, 5461, True),
    (8, 96, 256, 5462, False), (5, 193, 64, 8149, True), (5, 193, 64, 8150, False),
    (6, 129, 300, 6096, True), (6, 129, 300, 6097, False), (2, 193, 300, 16_299, True),
    (2, 193, 300, 16_300, False)])
def test_many_subspaces(gpu, dsub, m, ksub, n, small):
    """Around the row-subspaces past which the pruned searches take over (by
    sub-dimension and codewords)."""
    rng = np.random.default_rng(m + n)
    x = (rng.standard_normal((n, m * dsub)) * 0.2).astype(np.float32)
    cb = (rng.standard_normal((m, ksub, dsub)) * 0.2).astype(np.float32)
    device.profile_enable(True)
    device.profile_kernels(reset=True)
    got = _encode(x, cb, m, ksub)
    names = " ".join(device.profile_kernels(reset=True))
    device.profile_enable(False)
    assert ("encode_small_kernel" in names) == small
    assert np.array_equal(got, orc.pq_encode(x, m * dsub, m, ksub, cb, n_threads=8))


@pytest.mark.parametrize("dsub", [2, 4, 8])
@pytest.mark.parametrize("lanes", [4, 16])
def test_special_values_and_lane_count(gpu, dsub, lanes):
    """NaN, infinite and overflowing rows and codewords (a row with no distance
    below +inf gets code 0), at the reference hosts' lane counts."""
    m, ksub, n = 3, 200, 300
    rng = np.random.default_rng(dsub)
    x = (rng.standard_normal((n, m * dsub)) * 0.2).astype(np.float32)
    cb = (rng.standard_normal((m, ksub, dsub)) * 0.2).astype(np.float32)
    x[0, 0], x[1, :dsub], x[2, dsub], x[3] = np.nan, np.inf, -np.inf, 3e38
    cb[0, 0, 0], cb[0, 7, 1], cb[1, 5], cb[2, :, 0] = np.nan, np.inf, -3e38, np.nan
    with device.lanes(lanes), orc.lane_count(lanes):
        want = orc.pq_encode(x, m * dsub, m, ksub, cb, n_threads=8)
        assert np.array_equal(_encode(x, cb, m, ksub), want)
