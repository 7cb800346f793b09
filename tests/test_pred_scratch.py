"""The scratch of gpl_pred_noalloc, sized on the host: every model whose buffers for 64
test points fit the static array is taken, at every number of input columns."""

import ctypes as C

import pytest

from gplite_amd import _lib

FEAT = 64  # feature columns per model
SCRATCH = 64 << 20


def _align(b):
    return (b + 255) // 256 * 256


@pytest.mark.parametrize("ncols", [0, 1, 8, 59, 60, 61, 62, 128])
@pytest.mark.parametrize("M", [64, 128, 65600])
@pytest.mark.parametrize("N", [64, 4096, 65408, 65472])
def test_three_vectors_beside_the_matrices(N, M, ncols):
    f = getattr(_lib.lib(), "_ZN3gpl15pred_bufs_bytesElll")
    f.restype, f.argtypes = C.c_size_t, [C.c_int64] * 3
    want = _align(8 * M * max(ncols, 1)) + _align(8 * M * FEAT) + 2 * _align(8 * N * M) + _align(8 * M * 3)
    assert f(N, ncols, M) <= want


def test_largest_models_are_taken():
    f = getattr(_lib.lib(), "_ZN3gpl15pred_bufs_bytesElll")
    f.restype, f.argtypes = C.c_size_t, [C.c_int64] * 3
    assert f(65472, 61, 64) <= SCRATCH < f(65472, 62, 64)
