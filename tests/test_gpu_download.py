"""Host outputs at the edges of the staged download (5 MB, its chunks of at most
4 MB, its ring of four): decode round trips, and a bad code leaves `out` alone."""
import ctypes

import numpy as np
import pytest

from tac_gpu import errors, lib, pq

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("floats", [1, 524_287, 524_288, 524_289, 1_310_719, 1_310_720,
                                    1_310_721, 4_194_304, 4_194_305, 9_000_001])
def test_decode_sizes(gpu, floats):
    rng = np.random.default_rng(floats)
    cb = rng.standard_normal(256).astype(np.float32)
    codes = rng.integers(0, 256, (floats, 1)).astype(np.uint8)
    p = pq.PQ(dim=1, sub_dim=1, codebooks=cb, m=1)
    for _ in range(2):
        assert np.array_equal(p.decode_many(codes), cb[codes])


@pytest.mark.parametrize("n", [1_000_000, 2_000_000])
def test_bad_code_leaves_the_output(gpu, n):
    codes = np.zeros((n, 1), np.uint8)
    codes[-1] = 9
    out = np.full(n, 7.0, np.float32)
    cb = np.zeros(8, np.float32)

    def call():
        p = [a.ctypes.data_as(ctypes.c_void_p) for a in (codes, cb, out)]
        return lib.tac_pq_decode(p[0], n, 1, 1, 8, p[1], p[2])

    assert call() == errors.InvalidArgument.status and (out == 7.0).all()
    codes[-1] = 0
    assert call() == 0 and (out == 0.0).all()


@pytest.mark.parametrize("floats", [524_287, 1_310_721, 4_194_305, 9_000_001])
def test_pinned_output(gpu, floats):
    """Outputs inside a pinned allocation, from the runtime the library uses."""
    rng = np.random.default_rng(floats)
    cb = rng.standard_normal(256).astype(np.float32)
    codes = rng.integers(0, 256, (floats, 1)).astype(np.uint8)
    mem = ctypes.c_void_p()
    assert lib.hipHostMalloc(ctypes.byref(mem), ctypes.c_size_t(4 * (floats + 64)), 0) == 0
    try:
        out = np.ctypeslib.as_array(ctypes.cast(mem, ctypes.POINTER(ctypes.c_float)), (floats + 64,))

        def call(ksub):
            p = [ctypes.c_void_p(a.ctypes.data) for a in (codes, cb, out[32:])]
            return lib.tac_pq_decode(p[0], floats, 1, 1, ksub, p[1], p[2])

        for _ in range(2):
            out[:] = 7.0
            assert call(256) == 0
            assert np.array_equal(out[32:32 + floats], cb[codes[:, 0]])
            assert (out[:32] == 7.0).all() and (out[32 + floats:] == 7.0).all()
        out[:] = 7.0
        assert call(100) == errors.InvalidArgument.status and (out == 7.0).all()
    finally:
        del out
        lib.hipHostFree(mem)
