"""Frames whose resolution groups share their launches (all transforms of at most 512 points).

A context of one wavelength has a single group and takes the launches that larger frames take;
every scale of a many-level context must give the same maps, bit for bit, at sizes on and off
the transform lengths, in upright and wide frames, at sizes where all groups are merged and
where only the upper levels are.  One merged frame is also pinned against the FP64 oracle.
"""
import numpy as np
import pytest

import oracle_lib as O
from kpmatch import agreement, bits, rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def B():
    import bimp_amd
    if bimp_amd.device_count() < 1:
        pytest.fail("no GPU visible to the HIP library")
    return bimp_amd


def _bank(B):
    return B.make_lambdas_log(4, 64, 2)


@pytest.mark.parametrize("w,h", [(97, 161), (128, 128), (257, 130), (320, 240), (511, 513),
                                 (700, 90), (66, 600), (900, 520)])
def test_merged_scales_equal_single_ones(B, w, h):
    img = O.synth_frame(w, h, 20, w)
    lam = _bank(B)
    cs = B.CudaStuff(w, h, lam)
    cs.filter(img)
    cs.cells()
    for i, l in enumerate(sorted(lam)):
        one = B.CudaStuff(w, h, np.array([l], np.float32))
        one.filter(img)
        one.cells()
        for o in range(8):
            a = cs.get_map(i, B.MAP_COMPLEX, o)
            b = one.get_map(0, B.MAP_COMPLEX, o)
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), (i, o)
        for which in (B.MAP_DOUBLE, B.MAP_SINGLE):
            assert np.array_equal(cs.get_map(i, which).view(np.uint32),
                                  one.get_map(0, which).view(np.uint32)), (i, which)


@pytest.mark.parametrize("w,h", [(320, 240), (900, 520)])
def test_merged_frames_by_stream_and_graph(B, w, h):
    img = O.synth_frame(w, h, 25, 3)
    lam = _bank(B)
    orc = O.Oracle(w, h, lam)
    want, _, Ds, _ = orc.detect(img, cap=1 << 16, want_maps=True)
    cs = B.CudaStuff(w, h, lam)
    ref, n = cs.detect(img, cap=1 << 16)
    assert agreement(ref, want) >= 0.99
    assert max(rel_err(cs.get_map(i, B.MAP_DOUBLE), Ds[i]) for i in range(len(cs.ks))) <= 1e-4
    for flags in (B.FLAG_SINGLE_STREAM, B.FLAG_GRAPH, B.FLAG_GRAPH | B.FLAG_SINGLE_STREAM, 0):
        cs.set_flags(flags)
        for _ in range(2):
            got, m = cs.detect(img, cap=1 << 16)
            assert m == n and np.array_equal(bits(got), bits(ref))
    opt = B.default_options()
    opt.flags = B.FLAG_SINGLE_STREAM
    got, m = B.CudaStuff(w, h, lam, opt).detect(img, cap=1 << 16)
    assert m == n and np.array_equal(bits(got), bits(ref))
