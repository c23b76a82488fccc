"""Document layouts at the edges of the writer's slices (512 tokens) and scan
blocks (1,024 documents), against the oracle byte for byte."""
import numpy as np
import pytest

from oracle import binding as orc
from tac_gpu import device, errors, lib, storage

pytestmark = pytest.mark.gpu


def _check(lens, m, cb, seed=0):
    rng = np.random.default_rng(seed)
    off = np.concatenate([[3], 3 + np.cumsum(lens)]).astype(np.uint64)  # starts past token 0
    n = int(off[-1])
    a = rng.integers(0, 1 << 31, n).astype(np.uint32)
    codes = rng.integers(0, 256, (n, m)).astype(np.uint8 if cb == 1 else np.uint16)
    idx, pay = storage.write_doc_layouts(off, a, codes, m)
    st, ridx, rpay = orc.write_doc_layouts(off, a, codes, m, cb)
    assert st == 0 and np.array_equal(idx, ridx) and np.array_equal(pay, rpay)


@pytest.mark.parametrize("m,cb", [(16, 1), (21, 1), (1, 1), (5, 2), (16, 2)])
def test_slice_edges(gpu, m, cb):
    _check([511, 512, 513, 0, 1023, 1024, 1025, 1, 5000, 0], m, cb)


@pytest.mark.parametrize("lens", [[100_001], [600] * 40, [0] * 1023 + [700], [0] * 1024 + [700, 1],
                                  [2] * 1025 + [1537] * 3 + [1] * 2000])
def test_slices_and_scan_blocks(gpu, lens):
    _check(lens, 16, 1, seed=len(lens))


@pytest.mark.parametrize("n_docs", [32_767, 32_768, 65_537, 131_073, 262_143, 262_144, 300_007])
def test_groups_of_documents(gpu, n_docs):
    """1 to 16 documents a wave (by 32,768, 65,536, 131,072 and 262,144), the
    last group ragged, with documents around the slices' 512 tokens among them."""
    rng = np.random.default_rng(n_docs)
    lens = rng.integers(0, 4, n_docs)
    lens[rng.integers(0, n_docs, 60)] = rng.integers(500, 1030, 60)
    lens[[0, 15, 16, -2, -1]] = [512, 513, 600, 513, 512]
    _check(lens, 5, 1, seed=n_docs)


def test_layout_errors_leave_the_state_clean(gpu):
    """A short payload and unsound offsets with long documents, then a good call."""
    n = 3000
    a, c = np.zeros(n, np.uint32), np.zeros((n, 4), np.uint8)
    d_a, d_c = device.DeviceArray.from_host(a), device.DeviceArray.from_host(c)
    d_i, d_p = device.DeviceArray((4,), np.uint64), device.DeviceArray((40_000,), np.uint8)

    def call(off, payload):
        d_o = device.DeviceArray.from_host(np.array(off, np.uint64))
        return lib.tac_write_doc_layouts_device(d_o.ptr, len(off) - 1, n, d_a.ptr, d_c.ptr, 4, 1,
                                                d_i.ptr, d_p.ptr, payload, None)

    for _ in range(2):
        assert call([0, 2000, 3000], 100) == errors.BufferTooSmall.status
        assert call([0, 2000, 1000, 3000], 40_000) == errors.InvalidArgument.status
        assert call([0, 2900, 3001], 40_000) == errors.InvalidArgument.status
        assert call([0, 2000, 3000], 40_000) == 0
    _check([2000, 1000], 4, 1)
