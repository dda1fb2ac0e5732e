"""Every pyramid level against the oracle's, byte for byte: levels computed together by tiles, so
at sizes around the tile edges, at odd sizes and tiny ones (where the border reflects more than
once), one to six upper levels, both roundings, and frames at odd addresses and pitches.
"""
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


def _levels(img, n, half_up):
    out = [img]
    for _ in range(n):
        out.append(O.pyr_down(out[-1], half_up=half_up))
    return out


@pytest.mark.parametrize("w,h", [(16, 16), (17, 33), (64, 64), (65, 127), (128, 129), (350, 467),
                                 (513, 255), (1237, 701), (2049, 300), (300, 2047)])
@pytest.mark.parametrize("top", [8.0, 16.0, 32.0, 64.0, 128.0])
@pytest.mark.parametrize("half_up", [False, True])
def test_levels(B, w, h, top, half_up):
    lam = np.array([4.0, top], np.float32)
    if top > min(w, h):
        lam = lam[:1] * 2  # the frame is too small for this wavelength: one upper level
    cs = B.CudaStuff(w, h, lam)
    if half_up:
        cs.set_flags(B.FLAG_RESIZE_CPU)
    n = max(cs.ks[i].level for i in range(len(cs.ks)))
    rng = np.random.RandomState(w * 7 + h)
    img = rng.randint(0, 256, (h, w)).astype(np.uint8)
    img[: h // 3] = np.where(img[: h // 3] < 128, 0, 255)  # sums at both ends of the range
    cs.filter(img)
    for l, want in enumerate(_levels(img, n, half_up)):
        if l:
            assert np.array_equal(cs.get_level(l), want), (l, n)


def test_device_frame_at_odd_address_and_pitch(B):
    import torch
    w, h, pitch = 333, 251, 341
    lam = np.array([4.0, 32.0], np.float32)
    cs = B.CudaStuff(w, h, lam)
    rng = np.random.RandomState(5)
    buf = rng.randint(0, 256, pitch * h + 3).astype(np.uint8)
    dev = torch.from_numpy(buf).cuda()[3:]
    img = np.ascontiguousarray(buf[3:].reshape(h, pitch)[:, :w])
    assert B.lib.bimp_filter_u8(cs.ctx, dev.data_ptr(), pitch, 1, None) == 0
    torch.cuda.synchronize()
    n = max(cs.ks[i].level for i in range(len(cs.ks)))
    assert n >= 2
    for l, want in enumerate(_levels(img, n, False)):
        if l:
            assert np.array_equal(cs.get_level(l), want), l
