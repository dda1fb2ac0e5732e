"""Keypoint records that come back with the count: as many as the output holds, none beyond, and
frames with more of them than the context's pinned memory, bit for bit the device's records."""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

EARLY = 8192  # records that take no copy of their own


@pytest.fixture(scope="module")
def B():
    import bimp_amd
    if bimp_amd.device_count() < 1:
        pytest.fail("no GPU visible to the HIP library")
    return bimp_amd


def _noise(w, h, seed):
    return np.random.RandomState(seed).randint(0, 256, (h, w)).astype(np.uint8)


@pytest.mark.parametrize("w,h,bank,few", [(64, 48, 1, True), (320, 240, 8, True),
                                          (700, 520, 8, False)])
def test_records_at_every_capacity(B, w, h, bank, few):
    import torch
    cs = B.CudaStuff(w, h, O.BASE_BANK[:bank])
    img = _noise(w, h, w)
    full = torch.zeros((1 << 16, 7), dtype=torch.float32, device="cuda")
    n = C.c_int(-1)
    assert B.lib.bimp_detect_u8(cs.ctx, img.ctypes.data, w, 0, full.data_ptr(), 1 << 16, 1,
                                C.byref(n), None) == 0
    total = n.value
    assert (0 < total < EARLY) if few else (EARLY < total <= 1 << 16)
    want = full.cpu().numpy()[:total].view(np.uint32)
    for cap in (0, 1, total - 1, total, total + 1, EARLY - 1, EARLY, EARLY + 1, 1 << 16):
        out = np.full((cap + 4, 7), -3.0, np.float32)
        n = C.c_int(-1)
        st = B.lib.bimp_detect_u8(cs.ctx, img.ctypes.data, w, 0, out.ctypes.data, cap, 0,
                                  C.byref(n), None)
        assert n.value == total and (st == 0) == (total <= cap) and st >= 0
        m = min(total, cap)
        assert np.array_equal(out[:m].view(np.uint32), want[:m])
        assert np.all(out[m:] == -3.0)


@pytest.mark.parametrize("flags", ["", "FLAG_GRAPH", "FLAG_SINGLE_STREAM"])
def test_counts_follow_the_frames(B, flags):
    """Every call returns its own frame's count, an empty frame's included."""
    w, h = 200, 150
    cs = B.CudaStuff(w, h, O.BASE_BANK[:4])
    if flags:
        cs.set_flags(getattr(B, flags))
    frames = [_noise(w, h, 1), np.zeros((h, w), np.uint8), O.synth_frame(w, h, 10, 3)]
    ref = [B.CudaStuff(w, h, O.BASE_BANK[:4]).detect(f) for f in frames]
    for _ in range(3):
        for f, (kp, n) in zip(frames, ref):
            got, m = cs.detect(f)
            assert m == n
            assert np.array_equal(np.ascontiguousarray(got).view(np.uint8),
                                  np.ascontiguousarray(kp).view(np.uint8))
