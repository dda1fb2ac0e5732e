"""Two-nearest-neighbour matching into memory other than this device's, and in a captured graph.

Whole-number rows keep every FP32 sum exact, so indices equal the oracle's FP64 ones everywhere,
and distances its rounded square roots.
"""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

NQ, NT, DIM = 517, 433, 20


@pytest.fixture(scope="module")
def B():
    import bimp_amd
    if bimp_amd.device_count() < 1:
        pytest.fail("no GPU visible to the HIP library")
    return bimp_amd


@pytest.fixture(scope="module")
def data():
    import torch
    rng = np.random.default_rng(3)
    q = rng.integers(0, 4, (NQ, DIM)).astype(np.float32)
    t = rng.integers(0, 4, (NT, DIM)).astype(np.float32)
    t[NT // 2:] = t[: NT - NT // 2]  # every train row twice
    return torch.from_numpy(q).cuda(), torch.from_numpy(t).cuda(), O.knn2(q, t)


def _match(B, q, t, idx, dist, stream=None):
    st = B.lib.bimp_match_knn2(C.c_void_p(q.data_ptr()), NQ, DIM, C.c_void_p(t.data_ptr()), NT, DIM,
                               DIM, C.c_void_p(idx.data_ptr()), C.c_void_p(dist.data_ptr()), stream)
    assert st == B.OK


def _check(idx, dist, want):
    oi, od = want
    assert np.array_equal(idx.cpu().numpy(), oi)
    assert np.allclose(dist.cpu().numpy(), od, rtol=2.0 ** -22, atol=0)  # one rounded square root


@pytest.mark.parametrize("idx_host,dist_host", [(True, True), (True, False), (False, True)])
def test_outputs_in_pinned_host_memory(B, data, idx_host, dist_host):
    import torch
    q, t, want = data

    def out(dtype, host):
        return torch.full((NQ, 2), -7, dtype=dtype, **({"pin_memory": True} if host
                                                       else {"device": "cuda"}))
    idx, dist = out(torch.int32, idx_host), out(torch.float32, dist_host)
    torch.cuda.synchronize()
    _match(B, q, t, idx, dist)
    torch.cuda.synchronize()
    _check(idx, dist, want)


def test_replayed_in_a_graph(B, data):
    import torch
    q, t, want = data
    idx = torch.empty((NQ, 2), dtype=torch.int32, device="cuda")
    dist = torch.empty((NQ, 2), device="cuda")
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=side):
        _match(B, q, t, idx, dist, side.cuda_stream)
    for _ in range(3):
        idx.fill_(-7)
        dist.fill_(-7)
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        _check(idx, dist, want)
