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


def _backward(B, d, imgs, up):
    x, g, out = (B.DeviceBuffer(a.nbytes) for a in (imgs, up, imgs))
    x.upload(imgs)
    g.upload(up)
    gp = d.backward(x.ptr.value, len(imgs), g.ptr.value, out.ptr.value)
    return out.download(np.zeros_like(imgs)), gp


# frames that fill the padded array or not, with wavefronts inside every tap's reach and without,
# in launches that fill all 32 pairs; the reference gradient of one image pins the branch bits
@pytest.mark.parametrize("w,h,n", [(256, 256, 8), (512, 128, 8), (300, 256, 3), (320, 200, 2)])
def test_backward_inside_and_at_the_edges(B, w, h, n):
    from diff_ref import DiffRef
    lam = O.BASE_BANK[:4]
    imgs = np.stack([O.synth_frame(w, h, 15, 40 + i) for i in range(n)]).astype(np.float32)
    imgs /= np.float32(255)
    d = B.Diff(w, h, lam)
    up = np.random.default_rng(2).standard_normal((n, d.response_size)).astype(np.float32)
    ref = DiffRef(w, h, lam)
    targets = ref.forward(imgs[-1].astype(np.float64), gamma=0.6)
    _, rg, rp = ref.gradient(imgs[-1].astype(np.float64), targets)
    up[-1] = np.concatenate([2 * (a - b).ravel() for a, b in
                             zip(ref.forward(imgs[-1].astype(np.float64)), targets)])
    gi, _ = _backward(B, d, imgs, up)
    for i in range(n):
        one, gp = _backward(B, d, imgs[i:i + 1], up[i:i + 1])
        assert np.array_equal(gi[i].view(np.uint32), one[0].view(np.uint32)), i
    # the bars of the form's own gradient tests
    assert np.linalg.norm(one[0] - rg) <= 1e-3 * np.linalg.norm(rg)
    assert np.all(np.abs(gp - rp) <= 1e-3 * np.abs(rp))
