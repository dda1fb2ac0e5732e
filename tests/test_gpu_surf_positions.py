"""SURF descriptors of keypoints beyond the integers' range: pixels outside the frame count as 0, so
all their samples do, and the keypoints beside them in the list are not affected.
"""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


# a short list and a long one (two and four keypoints per workgroup)
@pytest.mark.parametrize("n", [16, 6002])
@pytest.mark.parametrize("upright", [True, False])
def test_positions_beyond_the_integers(n, upright):
    import bimp_amd as B
    w, h = 200, 150
    rng = np.random.default_rng(n)
    gray = O.synth_frame(w, h, 20, 1)
    mat = np.zeros((7, n), np.float32)
    mat[0], mat[1] = rng.uniform(20, w - 20, n), rng.uniform(20, h - 20, n)
    mat[4] = rng.uniform(5, 30, n)
    inside, _ = B.surf_descriptors(gray, mat, upright=upright)
    far = np.arange(n) % 2 == 1
    out = mat.copy()
    values = np.float32([np.inf, -np.inf, 3e9, -3e9, 2147483520.0])
    out[0, far] = values[np.arange(far.sum()) % 5]
    half = np.flatnonzero(far)[far.sum() // 2:]
    out[0, half], out[1, half] = mat[0, half], out[0, half]  # the other axis
    desc, ang = B.surf_descriptors(gray, out, upright=upright)
    assert np.all(desc[far] == 0) and np.all(ang[far] == 0)
    assert np.array_equal(desc[~far].view(np.uint32), inside[~far].view(np.uint32))
