"""Integral image, gray conversion and descriptors at the edges of their launches.

Integral image and gray conversion: whole numbers, equal to numpy's.  SURF and colour
descriptors: a keypoint's do not depend on the list it is in, bit for bit, so short lists and
lists on both sides of the split between the two launch shapes agree row by row (their values
are pinned against the oracle in test_gpu_features.py).
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


# bands of 4 rows, chunks of 2048 pixels, words of 4; 129 bands and more walk several per run
@pytest.mark.parametrize("w,h,pitch,shift", [(1, 1, 1, 0), (3, 4, 3, 1), (5, 5, 8, 0), (64, 3, 64, 0),
                                             (2047, 9, 2048, 0), (2049, 8, 2052, 0),
                                             (4100, 7, 4101, 0), (37, 517, 40, 2), (250, 130, 252, 0)])
def test_integral_edges(B, w, h, pitch, shift):
    rng = np.random.default_rng(w + h)
    buf = rng.integers(0, 256, shift + h * pitch, dtype=np.uint8)
    img = buf[shift:].reshape(h, pitch)[:, :w]
    d, out = B.DeviceBuffer(buf.nbytes), B.DeviceBuffer(4 * (w + 1) * (h + 1))
    d.upload(buf)
    got = np.full((h + 1, w + 1), 0xdeadbeef, np.uint32)
    out.upload(got)
    assert B.lib.bimp_integral_image(C.c_void_p(d.ptr.value + shift), pitch, w, h, out.ptr,
                                     None) == B.OK
    out.download(got)
    want = np.zeros((h + 1, w + 1), np.uint32)
    want[1:, 1:] = img.astype(np.uint32).cumsum(0).cumsum(1)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("w,h,bpitch,gpitch,shift", [(1, 1, 3, 1, 0), (5, 3, 15, 5, 0),
                                                     (8, 2, 24, 8, 0), (513, 2, 1540, 516, 0),
                                                     (515, 3, 1548, 516, 1)])
def test_gray_edges(B, w, h, bpitch, gpitch, shift):
    rng = np.random.default_rng(w)
    buf = rng.integers(0, 256, shift + h * bpitch, dtype=np.uint8)
    v = buf[shift:].reshape(h, bpitch)[:, :3 * w].reshape(h, w, 3).astype(np.uint32)
    want = ((1868 * v[..., 0] + 9617 * v[..., 1] + 4899 * v[..., 2] + (1 << 13)) >> 14)
    d, out = B.DeviceBuffer(buf.nbytes), B.DeviceBuffer(h * gpitch)
    d.upload(buf)
    got = np.full((h, gpitch), 77, np.uint8)
    out.upload(got)
    assert B.lib.bimp_bgr_to_gray(C.c_void_p(d.ptr.value + shift), bpitch, w, h, 1, out.ptr,
                                  gpitch, None) == B.OK
    out.download(got)
    assert np.array_equal(got[:, :w], want)
    assert np.all(got[:, w:] == 77)


@pytest.mark.parametrize("upright", [False, True])
def test_descriptors_do_not_depend_on_the_list(B, upright):
    w, h, n = 320, 200, 6003
    gray = O.synth_frame(w, h, 30, 3)
    rng = np.random.default_rng(0)
    bgr = rng.integers(0, 256, (h, w, 3), dtype=np.uint8)
    mat = np.zeros((7, n), np.float32)
    mat[0], mat[1] = rng.uniform(-4, w + 4, n), rng.uniform(-4, h + 4, n)
    mat[4] = O.BASE_BANK[rng.integers(0, 8, n)] * rng.choice([1, 4], n)
    desc, ang = B.surf_descriptors(gray, mat, upright=upright)
    col = B.color_features(mat, bgr)
    for lo, hi in ((0, 1), (1, 3), (3, 6), (6, 13), (20, 5999), (n - 5, n)):
        d, a = B.surf_descriptors(gray, mat[:, lo:hi], upright=upright)
        assert np.array_equal(d.view(np.uint32), desc[lo:hi].view(np.uint32))
        assert np.array_equal(a.view(np.uint32), ang[lo:hi].view(np.uint32))
        c = B.color_features(np.ascontiguousarray(mat[:, lo:hi]), bgr)
        assert np.array_equal(c.view(np.uint32), col[lo:hi].view(np.uint32))
