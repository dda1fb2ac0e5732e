"""Two-nearest-neighbour matching at the edges of its tiles, slices and alignment rules.

Whole-number rows keep every FP32 sum exact, so indices (ties included: the lower train index
wins) equal the oracle's FP64 ones everywhere, and distances its rounded square roots.
"""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def B():
    import bimp_amd
    if bimp_amd.device_count() < 1:
        pytest.fail("no GPU visible to the HIP library")
    return bimp_amd


def _rows(rng, n, dim, ld):
    a = np.zeros((n, ld), np.float32)
    a[:, :dim] = rng.integers(0, 4, (n, dim))
    return a


# tiles of 32 and 64 rows; pieces of 16 dimensions; strides that are and are not multiples of
# four floats; outputs 8-byte aligned (slices meet in them) and only 4-byte aligned (one slice)
@pytest.mark.parametrize("nq,nt,dim,ld,shift", [
    (1, 1, 1, 1, 0), (33, 31, 15, 16, 0), (32, 64, 16, 16, 0), (31, 65, 17, 17, 0),
    (64, 129, 3, 5, 0), (40, 200, 64, 64, 1), (1, 2100, 33, 36, 0), (2100, 1, 8, 8, 0),
    (1790, 1795, 20, 20, 0), (1790, 1795, 7, 9, 0), (1790, 1795, 18, 20, 1),
])
def test_knn2_edges(B, nq, nt, dim, ld, shift):
    rng = np.random.default_rng(nq * 7 + nt * 3 + dim)
    q, t = _rows(rng, nq, dim, ld), _rows(rng, nt, dim, ld)
    t[nt // 2:] = t[: nt - nt // 2]  # every train row twice
    dq, dt = B.DeviceBuffer(q.nbytes), B.DeviceBuffer(t.nbytes)
    di, dd = B.DeviceBuffer(8 * nq + 8), B.DeviceBuffer(8 * nq + 8)
    dq.upload(q)
    dt.upload(t)
    st = B.lib.bimp_match_knn2(dq.ptr, nq, ld, dt.ptr, nt, ld, dim,
                               C.c_void_p(di.ptr.value + 4 * shift),
                               C.c_void_p(dd.ptr.value + 4 * shift), None)
    assert st == B.OK
    idx, dist = np.zeros(2 * nq + 2, np.int32), np.zeros(2 * nq + 2, np.float32)
    di.download(idx)
    dd.download(dist)
    idx = idx[shift: shift + 2 * nq].reshape(nq, 2)
    dist = dist[shift: shift + 2 * nq].reshape(nq, 2)
    oi, od = O.knn2(np.ascontiguousarray(q[:, :dim]), np.ascontiguousarray(t[:, :dim]))
    assert np.array_equal(idx, oi)
    fin = np.isfinite(od)
    assert np.array_equal(np.isfinite(dist), fin)
    assert np.allclose(dist[fin], od[fin], rtol=2.0 ** -22, atol=0)  # one rounded square root


def test_knn2_unusable_distances(B):
    """Rows at NaN distance are never neighbours, rows at infinite distance are after the finite
    ones; a query without a second row gets index -1 and +inf."""
    q = np.zeros((40, 4), np.float32)
    t = np.full((200, 4), np.nan, np.float32)
    t[150] = 1.0
    t[20] = np.inf
    idx, dist = B.match_knn2(q, t)
    assert np.array_equal(idx, np.tile([150, 20], (40, 1)))
    assert np.array_equal(dist, np.tile(np.float32([2.0, np.inf]), (40, 1)))
    idx, dist = B.match_knn2(q, t[:150][21:])
    assert np.all(idx == -1) and np.all(np.isinf(dist))
