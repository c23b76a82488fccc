"""refine at the edges of its kernel's tiles (64 and 128 document tokens, 64
query tokens, groups of 8 and 16 subspaces), against the oracle bit for bit."""
import ctypes

import numpy as np
import pytest

from oracle import binding as orc
from tac_gpu import device, errors, lib, retrieval

pytestmark = pytest.mark.gpu

LENS = [0, 1, 2, 31, 32, 33, 63, 64, 65, 127, 128, 129, 200, 0, 5]


# means of 1.2, 1.8 and 9.5 tokens: a wave a candidate past 512 or 1,024
SHORT = [1, 0, 1, 2, 1, 1, 2, 1, 1, 2]
SHORTER = [1, 2, 2, 2, 2, 2, 2, 1, 2, 2]
MIXED = [0, 1, 7, 8, 9, 15, 16, 17, 3, 2, 5, 4, 40, 6]


def _index(dim, m, ksub, n_q, seed=0, lens=LENS):
    rng = np.random.default_rng(seed + dim + m + n_q)
    off = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint64)
    n = int(off[-1])
    cents = rng.standard_normal((40, dim)).astype(np.float32)
    assign = rng.integers(0, 40, n).astype(np.uint32)
    codes = rng.integers(0, ksub, (n, m)).astype(np.uint8 if ksub <= 256 else np.uint16)
    st, idx, pay = orc.write_doc_layouts(off, assign, codes, m, codes.itemsize)
    assert st == 0
    norms = rng.random(n).astype(np.float32)
    table = rng.standard_normal(m * ksub * n_q).astype(np.float32)
    q = rng.standard_normal((n_q, dim)).astype(np.float32)
    return retrieval.DocIndex(dim, m, ksub, cents, idx, pay, off, norms), table, q


def _want(ix, table, q, n_q):
    out = np.empty(ix.n_docs, np.float32)
    for d in range(ix.n_docs):
        st, out[d] = orc.refine(q, n_q, ix.dim, ix.centroids, table, ix.m, ix.ksub, ix.doc_index,
                                ix.doc_payload, ix.doc_token_offsets, ix.residual_norms, d)
        assert st == 0
    return out


@pytest.mark.parametrize("dim,m,ksub,n_q", [
    (64, 16, 256, 32), (64, 32, 256, 8), (64, 8, 256, 64), (64, 16, 256, 65), (64, 16, 1024, 17),
    (128, 16, 256, 33), (128, 32, 256, 1), (128, 20, 200, 16), (63, 21, 256, 9), (96, 12, 256, 40),
    (64, 1, 3, 5), (2, 8200, 2, 2)])
@pytest.mark.parametrize("n_cand", [15, 600])
def test_refine_tile_edges(gpu, dim, m, ksub, n_q, n_cand):
    ix, table, q = _index(dim, m, ksub, n_q)
    want = _want(ix, table, q, n_q)
    cand = np.random.default_rng(1).integers(0, ix.n_docs, n_cand).astype(np.uint32)
    cand[:ix.n_docs] = np.arange(ix.n_docs)
    got = retrieval.refine(ix, table, q, n_q, cand)
    assert np.array_equal(got.view(np.uint32), want[cand].view(np.uint32))


@pytest.mark.parametrize("lens", [SHORT, SHORTER, MIXED])
@pytest.mark.parametrize("dim,m,ksub,n_q", [
    (64, 16, 256, 32), (64, 32, 256, 8), (64, 16, 1024, 65), (128, 16, 256, 33), (128, 20, 200, 1),
    (63, 21, 256, 9), (96, 12, 256, 40), (48, 3, 3, 64), (200, 25, 256, 3), (768, 96, 256, 4),
    (1536, 16, 256, 2), (1537, 1, 256, 2), (2, 1600, 2, 2)])
@pytest.mark.parametrize("n_cand", [512, 513, 1025, 70_001])
def test_refine_short_documents(gpu, lens, dim, m, ksub, n_q, n_cand):
    """A wave a candidate (four a block, 65,536 of the grid's at once), around
    the rules that choose it."""
    ix, table, q = _index(dim, m, ksub, n_q, lens=lens)
    want = _want(ix, table, q, n_q)
    cand = np.random.default_rng(2).integers(0, ix.n_docs, n_cand).astype(np.uint32)
    got = retrieval.refine(ix, table, q, n_q, cand)
    assert np.array_equal(got.view(np.uint32), want[cand].view(np.uint32))


@pytest.mark.parametrize("dim", [64, 96])
@pytest.mark.parametrize("where", ["code", "id", "count", "doc"])
def test_refine_short_documents_corrupt(gpu, dim, where):
    """The first failing candidate of many is reported, whichever wave meets it;
    a clean call works afterwards."""
    m, ksub, n_q, n_cand = 16, 200, 20, 3000
    ix, table, q = _index(dim, m, ksub, n_q, seed=5, lens=MIXED)
    bad, d = ix.doc_payload.copy(), 7  # 17 tokens
    lo = int(ix.doc_index[d])
    if where == "code":
        bad[lo + 4 + 4 * 17 + 17 * m - 1] = 250
    elif where == "id":
        bad[lo + 4 + 4 * 16] = 40
    elif where == "count":
        bad[lo] = 16
    ixb = retrieval.DocIndex(dim, m, ksub, ix.centroids, ix.doc_index, bad, ix.doc_token_offsets,
                             ix.residual_norms)
    cand = np.full(n_cand, 3, np.uint32)
    cand[[1234, 2900, 2999]] = ix.n_docs if where == "doc" else d
    kind = errors.DocOutOfRange if where == "doc" else errors.DocLayoutCorrupt
    with pytest.raises(kind):
        retrieval.refine(ixb, table, q, n_q, cand)
    assert lib.tac_gpu_last_error().endswith(b"candidate 1234")
    cand[:] = np.arange(n_cand) % ix.n_docs
    got = retrieval.refine(ix, table, q, n_q, cand)
    assert np.array_equal(got.view(np.uint32), _want(ix, table, q, n_q)[cand].view(np.uint32))


@pytest.mark.parametrize("shift", [1, 2, 4])
def test_refine_unaligned_device_arrays(gpu, shift):
    """Payload at any byte, centroids and queries at any float."""
    dim, m, ksub, n_q = 64, 16, 256, 20
    ix, table, q = _index(dim, m, ksub, n_q, seed=3)
    want = _want(ix, table, q, n_q)

    def put(a, by):
        raw = np.zeros(a.nbytes + 16, np.uint8)
        raw[by:by + a.nbytes] = np.ascontiguousarray(a).reshape(-1).view(np.uint8)
        d = device.DeviceArray.from_host(raw)
        keep.append(d)
        return ctypes.c_void_p(d.ptr.value + by)

    keep = []
    by4 = 4 if shift == 4 else 0
    view = retrieval._DocIndexC(dim, 40, m, ksub, ix.n_docs, ix.residual_norms.size,
                                ix.doc_payload.size, put(ix.centroids, by4),
                                put(ix.doc_index, 0), put(ix.doc_payload, shift),
                                put(ix.doc_token_offsets, 0), put(ix.residual_norms, by4))
    cand = np.arange(ix.n_docs, dtype=np.uint32)
    scores = device.DeviceArray((ix.n_docs,), np.float32)
    errors.check(lib.tac_refine_device(ctypes.byref(view), put(table, 0), table.size, put(q, by4),
                                       n_q, put(cand, 0), cand.size, scores.ptr, None))
    assert np.array_equal(scores.to_host().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("where", ["code", "count"])
def test_refine_corrupt_layouts(gpu, where):
    """A code past ksub in the last token, or a token count that is not the
    document's: DocLayoutCorrupt, and a clean call works afterwards."""
    dim, m, ksub, n_q = 64, 16, 200, 4
    ix, table, q = _index(dim, m, ksub, n_q, seed=5)
    bad = ix.doc_payload.copy()
    d = 11  # 129 tokens
    lo = int(ix.doc_index[d])
    if where == "code":
        bad[lo + 4 + 4 * 129 + 129 * m - 1] = 250
    else:
        bad[lo] = 128
    ixb = retrieval.DocIndex(dim, m, ksub, ix.centroids, ix.doc_index, bad, ix.doc_token_offsets,
                             ix.residual_norms)
    with pytest.raises(errors.DocLayoutCorrupt):
        retrieval.refine(ixb, table, q, n_q, [0, d, 3])
    got = retrieval.refine(ixb, table, q, n_q, [12, 3])
    assert np.array_equal(got.view(np.uint32), _want(ix, table, q, n_q)[[12, 3]].view(np.uint32))
