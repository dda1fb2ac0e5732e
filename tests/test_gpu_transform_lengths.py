"""Every transform length that 64 lanes hold, as row and as column length, against the FP64 oracle.

The first exchange of these transforms stays in registers for all but 1024 points, and the rest
of the frame's kernels read and write them at fixed places, so a wrong lane or register is an
error of the size of the map.  The tolerance: two FP32 transforms of up to 12 doublings round
by less than 24 * 2^-24 = 1.4e-6 of the largest response each, a response map sums about ten of
them: 2e-5.
"""
import numpy as np
import pytest

import oracle_lib as O
from kpmatch import rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def B():
    import bimp_amd
    if bimp_amd.device_count() < 1:
        pytest.fail("no GPU visible to the HIP library")
    return bimp_amd


# (the 7- and 3-row remainders leave the last row pair, row unit and staging round ragged)
@pytest.mark.parametrize("n,side", [(512, 307), (512, 470), (1024, 611), (1024, 515),
                                    (1536, 1155), (1536, 1043), (2048, 1601), (2560, 2115),
                                    (3072, 2627), (3584, 3139)])
@pytest.mark.parametrize("upright", [False, True])
def test_length(B, n, side, upright):
    other = 71
    w, h = (other, side) if upright else (side, other)
    lam = O.BASE_BANK[:1]
    cs = B.CudaStuff(w, h, lam)
    assert (cs.ks[0].fft_h if upright else cs.ks[0].fft_w) == n
    img = O.synth_frame(w, h, 30, n)
    _, _, Ds, Ss = O.Oracle(w, h, lam).detect(img, want_maps=True)
    cs.filter(img)
    cs.cells()
    for which, want in ((B.MAP_DOUBLE, Ds[0]), (B.MAP_SINGLE, Ss[0])):
        e = rel_err(cs.get_map(0, which), want)
        print(f"{w}x{h} map {which}: {e:.2e}", flush=True)
        assert np.isfinite(e) and e <= 2e-5
