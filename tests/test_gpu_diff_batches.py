"""Responses of several images at once equal those of each image alone, bit for bit: launches of
up to 32 (scale, image) pairs, at image counts that divide into them and that do not, groups of
one to eight scales, and images whose intermediates leave room for fewer pairs per launch.
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


def _forward(B, d, imgs):
    x, r = B.DeviceBuffer(imgs.nbytes), B.DeviceBuffer(4 * len(imgs) * d.response_size)
    x.upload(imgs)
    d.forward(x.ptr.value, len(imgs), r.ptr.value)
    return r.download(np.full((len(imgs), d.response_size), np.nan, np.float32))


@pytest.mark.parametrize("w,h,bank,n", [(128, 128, O.BASE_BANK[:1], 9), (131, 97, O.BASE_BANK, 8),
                                        (131, 97, O.BASE_BANK, 17), (96, 130, O.BASE_BANK[:3], 11),
                                        (333, 251, O.BASE_BANK, 5), (640, 500, O.BASE_BANK, 3)])
def test_batch_equals_single_images(B, w, h, bank, n):
    imgs = np.stack([O.synth_frame(w, h, 15, i) for i in range(n)]).astype(np.float32)
    imgs /= np.float32(255)
    d = B.Diff(w, h, np.asarray(bank, np.float32))
    got = _forward(B, d, imgs)
    one = np.concatenate([_forward(B, B.Diff(w, h, np.asarray(bank, np.float32)), imgs[i:i + 1])
                          for i in range(n)])
    assert np.all(np.isfinite(one))
    assert np.array_equal(got.view(np.uint32), one.view(np.uint32))
