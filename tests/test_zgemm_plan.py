"""How the batched product is cut into launches (host code, no GPU): every
launch within HIP's limits (fewer than 2^32 threads along x, at most 65535
products along z) up to the largest sizes that are accepted, and the 64 x 128
tiles for the sizes that the product tests take for them."""

import ctypes

import pytest

from mrmustard_amd import _lib

CU = 256
TOP = ((1 << 24) - 1) * 128  # columns of the widest product


def _plan(M, N, batch, shared, rc=_lib.MM_OK):
    out = (ctypes.c_int64 * 4)()
    assert _lib.load().mm_zgemm_plan(M, N, batch, shared, CU, ctypes.addressof(out)) == rc
    return tuple(out)


@pytest.mark.parametrize("shared", [0, 1])
@pytest.mark.parametrize("M,N,batch", [
    (1, 1, 1), (4, 1 << 30, 1), (4, (1 << 30) - 64, 1), (4, (1 << 30) - 63, 1), (64, TOP, 1), (100, TOP, 2), (16, 1 << 29, 3),
    (2, 1024, 1 << 20), (2, 1 << 20, 1 << 10), (2, 1 << 20, 1023), (3, 7, 1 << 32), (2, (1 << 29) - 32, 5), (2, (1 << 29) - 31, 5),
    (1000, 70000, 70000), (700, 1 << 30, 2),
])
def test_launches_within_limits(M, N, batch, shared):
    rt, step, cols, merged = _plan(M, N, batch, shared)
    wide = cols * step if merged else cols
    blocks = -(-wide // (64 if rt else 128))
    assert 1 <= step <= batch and 1 <= cols <= N and (cols == N or not merged)
    assert blocks * 256 < 1 << 32
    assert merged or step <= 65535
    assert -(-M // (16 * rt if rt else 64)) <= 65535
    assert rt or cols == N


def test_shared_products_stay_merged():
    assert _plan(10, 100, 700, 1)[1:] == (700, 100, 1)
    assert _plan(100, 100, 10000, 1)[1:] == (10000, 100, 1)
    assert _plan(10, 100, 700, 0)[1:] == (700, 100, 0)


def test_too_large_is_refused():
    _plan(1, TOP + 1, 1, 0, _lib.MM_ERR_UNSUPPORTED)
    _plan(65535 * 64 + 1, 1, 1, 0, _lib.MM_ERR_UNSUPPORTED)
