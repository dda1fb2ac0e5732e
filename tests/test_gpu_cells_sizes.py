"""The cells stage at sizes whose transform is as wide or as high as the data (column W and row H
wrap around there): bit-exact against the oracle on the oracle's complex maps, with tiles on the
unchecked and the checked path."""
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


# interior tiles of 64 x 16 end at the last column or row that does not wrap: widths and heights
# that are, and just are not, transform lengths
@pytest.mark.parametrize("w,h", [(256, 256), (256, 100), (300, 128), (128, 512), (255, 256),
                                 (512, 64)])
def test_cells_bit_exact_at_transform_sizes(B, w, h):
    lam = O.BASE_BANK
    cs, orc = B.CudaStuff(w, h, lam), O.Oracle(w, h, lam)
    orc.set_image(O.synth_frame(w, h, 15, w + h))
    for i, si in enumerate(cs.ks):
        maps = orc.filter(i)
        for o in range(8):
            cs.set_map(i, B.MAP_COMPLEX, maps[o, :si.map_h, :si.map_w], o)
        D, S = orc.cells(i, maps)
        cs.cells()
        assert np.array_equal(cs.get_map(i, B.MAP_DOUBLE).view(np.uint32), D.view(np.uint32)), i
        assert np.array_equal(cs.get_map(i, B.MAP_SINGLE).view(np.uint32), S.view(np.uint32)), i
