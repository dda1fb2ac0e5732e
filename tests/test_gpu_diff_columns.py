"""Gradients of the differentiation form with column transforms above 512 points, and with a group
of scales that does not fit one backward launch.

The column kernels of the backward change form with the length: the sum over orientations leaves the
registers from 1536 points on, blocks narrow to four columns above 2048, and 4096 points take two
wavefronts.  Tall narrow images reach each of them; image and parameter gradients against the
FP64 reference gradient (tests/diff_ref.py) with the bars of the form's own tests.
"""
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


# columns of 1024, 1536, 2048, 2560, 3072, 3584 and 4096 points, padded and (1024) full; two scales at
# level 0 and one at level 1
@pytest.mark.parametrize("h", [700, 1024, 1155, 1601, 2115, 2601, 3111, 3700])
def test_gradients_of_tall_images(B, h):
    w, lam = 72, O.BASE_BANK[[0, 3, 5]]
    img = O.synth_frame(w, h, 40, h).astype(np.float32) / np.float32(255)
    ref = DiffRef(w, h, lam)
    x = img.astype(np.float64)
    targets = ref.forward(x, gamma=0.6)
    _, rg, rp = ref.gradient(x, targets)
    up = np.concatenate([2 * (a - b).ravel() for a, b in zip(ref.forward(x), targets)])
    d = B.Diff(w, h, lam)
    gi, gp = _backward(B, d, img[None], up[None].astype(np.float32))
    ei = np.linalg.norm(gi[0] - rg) / np.linalg.norm(rg)
    print(f"{w}x{h}: image {ei:.1e}, parameters {np.abs(gp - rp) / np.abs(rp)}", flush=True)
    assert ei <= 1e-3
    assert np.all(np.abs(gp - rp) <= 1e-3 * np.abs(rp))


def test_group_larger_than_a_launch(B):
    """Eight scales of one level whose buffers hold seven at a time: parameters are set and the
    gradient taken in two parts.  Responses equal those of one context per scale bit for bit; the
    image gradient is their sum, rounded at most twice per scale."""
    w, h = 1600, 1100  # 2048 x 1536 padded: 579 MB of work buffers per scale, 4 GB in all
    lam = np.linspace(4, 7.4, 8).astype(np.float32)
    img = O.synth_frame(w, h, 100, 3).astype(np.float32)[None] / np.float32(255)
    x = B.DeviceBuffer(img.nbytes)
    x.upload(img)
    d = B.Diff(w, h, lam)
    up = np.random.default_rng(4).standard_normal((1, d.response_size)).astype(np.float32)
    out = B.DeviceBuffer(4 * d.response_size)
    d.forward(x.ptr.value, 1, out.ptr.value)
    resp = out.download(np.zeros(d.response_size, np.float32))
    gi, gp = _backward(B, d, img, up)
    d.close()
    n = w * h
    total, size, ps = np.zeros((h, w)), np.zeros((h, w)), []
    for k in range(8):
        one = B.Diff(w, h, lam[k:k + 1])
        o1 = B.DeviceBuffer(4 * n)
        one.forward(x.ptr.value, 1, o1.ptr.value)
        r1 = o1.download(np.zeros(n, np.float32))
        assert np.array_equal(r1.view(np.uint32), resp[k * n:(k + 1) * n].view(np.uint32)), k
        g1, p1 = _backward(B, one, img, np.ascontiguousarray(up[:, k * n:(k + 1) * n]))
        one.close()
        total += g1[0]
        size += np.abs(g1[0])
        ps.append(p1)
    assert np.all(np.abs(gi[0] - total) <= 16 * 2.0 ** -24 * size)
    assert np.allclose(gp, np.sum(ps, axis=0), rtol=0, atol=1e-9 * np.abs(ps).sum())
