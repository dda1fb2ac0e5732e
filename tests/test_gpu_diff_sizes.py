"""Gradients of the differentiation form over the shapes its backward launches divide by.

Image and parameter gradients against the FP64 reference gradient (tests/diff_ref.py) at sizes
with and without padding, odd sides, transforms of 64 to 512 points and of two lengths at once;
and batches whose images do not divide into the launches, equal to their images one by one.
The bars are those of the form's own tests (1e-3, FP32 against FP64 branch decisions).
"""
import ctypes as C

import numpy as np
import pytest

import oracle_lib as O
from diff_ref import DiffRef

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def B():
    import bimp_amd
    if bimp_amd.device_count() < 1:
        pytest.fail("no GPU visible to the HIP library")
    return bimp_amd


def _backward(B, d, imgs, up):
    x, g, out = (B.DeviceBuffer(a.nbytes) for a in (imgs, up, imgs))
    x.upload(imgs)
    g.upload(up)
    gp = d.backward(x.ptr.value, len(imgs), g.ptr.value, out.ptr.value)
    return out.download(np.zeros_like(imgs)), gp


# widths and heights on, just below and just above transform lengths; a four-scale and an
# eight-scale bank (the latter on two pyramid levels)
@pytest.mark.parametrize("w,h,scales", [(128, 128, 4), (129, 64, 4), (255, 130, 8), (200, 257, 4),
                                        (131, 512, 4), (256, 256, 8)])
def test_gradients_over_sizes(B, w, h, scales):
    lam = O.BASE_BANK[:scales]
    img = O.synth_frame(w, h, 12, w + h).astype(np.float32) / np.float32(255)
    ref = DiffRef(w, h, lam)
    x = img.astype(np.float64)
    targets = ref.forward(x, gamma=0.6)
    _, rg, rp = ref.gradient(x, targets)
    up = np.concatenate([2 * (a - b).ravel() for a, b in zip(ref.forward(x), targets)])
    d = B.Diff(w, h, lam)
    gi, gp = _backward(B, d, img[None], up[None].astype(np.float32))
    assert np.linalg.norm(gi[0] - rg) <= 1e-3 * np.linalg.norm(rg)
    assert np.all(np.abs(gp - rp) <= 1e-3 * np.abs(rp))


@pytest.mark.parametrize("w,h,n", [(128, 128, 9), (150, 133, 11)])
def test_batch_equals_single_images(B, w, h, n):
    lam = O.BASE_BANK
    imgs = np.stack([O.synth_frame(w, h, 12, i) for i in range(n)]).astype(np.float32)
    imgs /= np.float32(255)
    d = B.Diff(w, h, lam)
    up = np.random.default_rng(1).standard_normal((n, d.response_size)).astype(np.float32)
    gi, gp = _backward(B, d, imgs, up)
    ps = np.zeros(2)
    for i in range(n):
        one, p1 = _backward(B, d, imgs[i:i + 1], up[i:i + 1])
        assert np.array_equal(one[0].view(np.uint32), gi[i].view(np.uint32))
        ps += p1
    # the library adds the images' partial sums one by one in double
    assert np.allclose(gp, ps, rtol=1e-9, atol=1e-9 * np.abs(ps).max())


# 841, 1089 and 2809 taps: below, just above and above two of the chunks the sums walk
@pytest.mark.parametrize("lam", [4.0, 4.6, 7.4])
def test_bank_of_new_parameters(B, lam):
    """Responses after a parameter change equal those of a context created with the parameters,
    bit for bit, and the FP64 restatement's within the form's 1e-4."""
    w, h, ratio, gamma = 130, 96, 0.61, 0.45
    lams = np.array([lam], np.float32)
    img = O.synth_frame(w, h, 12, 5).astype(np.float32)[None] / np.float32(255)
    opt = B.default_options()
    opt.sigma_ratio, opt.gamma = ratio, gamma
    x = B.DeviceBuffer(img.nbytes)
    x.upload(img)
    got = []
    for d in (B.Diff(w, h, lams), B.Diff(w, h, lams, opt)):
        d.set_params(ratio, gamma)
        out = B.DeviceBuffer(4 * d.response_size)
        d.forward(x.ptr.value, 1, out.ptr.value)
        got.append(out.download(np.zeros(d.response_size, np.float32)))
    assert np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))
    ref = np.concatenate([r.ravel() for r in DiffRef(w, h, lams).forward(
        img[0].astype(np.float64), ratio=float(np.float32(ratio)), gamma=float(np.float32(gamma)))])
    assert np.abs(got[0] - ref).max() <= 1e-4 * np.abs(ref).max()
