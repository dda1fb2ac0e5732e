"""SURF on an integral image of more than 2^30 entries, whose byte offsets pass 32 bits: the same
content in the far corner of such a frame and in a small frame gives the same bits.  Scale 2 keeps
every sample position whole (upright; an oriented list, its angles)."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


def test_integral_beyond_32_bit_offsets():
    import torch
    import bimp_amd as B
    n, W, H, k = 256, 32800, 32768, 40
    assert (W + 1) * (H + 1) > 1 << 30
    rng = np.random.default_rng(8)
    img = torch.from_numpy(O.synth_frame(n, n, 30, 2)).cuda()
    small = torch.empty((n + 1, n + 1), dtype=torch.int32, device="cuda")
    big = torch.zeros((H + 1, W + 1), dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    assert B.lib.bimp_integral_image(C.c_void_p(img.data_ptr()), n, n, n,
                                     C.c_void_p(small.data_ptr()), None) == B.OK
    big[H - n:, W - n:] = small
    kp = np.zeros((7, k), np.float32)
    kp[0], kp[1] = rng.integers(0, n, k), rng.integers(0, n, k)  # some reach past the edges
    kp[4] = 15.0
    assert np.float32(1.2) * np.float32(15) / np.float32(9) == 2
    for upright in (1, 0):
        got = []
        for ii, w, h, ox, oy in ((small, n, n, 0, 0), (big, W, H, W - n, H - n)):
            m = kp.copy()
            m[0] += ox
            m[1] += oy
            mat = torch.from_numpy(m).cuda()
            desc = torch.full((k, 64), -7.0, device="cuda")
            ang = torch.full((k,), -7.0, device="cuda")
            torch.cuda.synchronize()
            assert B.lib.bimp_surf_descriptors(
                C.c_void_p(ii.data_ptr()), w, h, C.c_void_p(mat.data_ptr()), k, k, upright,
                C.c_void_p(desc.data_ptr()), 64, C.c_void_p(ang.data_ptr()), None) == B.OK
            torch.cuda.synchronize()
            got.append((desc.cpu().numpy(), ang.cpu().numpy()))
        (ds, as_), (db, ab) = got
        assert np.array_equal(as_.view(np.uint32), ab.view(np.uint32))
        if upright:
            assert np.array_equal(ds.view(np.uint32), db.view(np.uint32))
            assert np.allclose(np.linalg.norm(db, axis=1), 1, atol=1e-5)
