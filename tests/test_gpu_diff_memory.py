"""Device memory of a differentiation context: work buffers for the (scale, image) pairs that its
launches can hold, and no more."""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scales", [1, 2])
def test_context_memory(scales):
    import torch
    import bimp_amd as B
    w, h = 512, 512
    B.Diff(w, h, O.BASE_BANK[:1]).close()  # kernels loaded, allocator warm
    torch.cuda.synchronize()
    free0 = torch.cuda.mem_get_info()[0]
    d = B.Diff(w, h, O.BASE_BANK[:scales])
    used = free0 - torch.cuda.mem_get_info()[0]
    pixels = w * h  # a power of two: no padding
    # eight images per scale at 184 bytes and 8 tap rows of 55 columns at most; the forward's
    # spectra and maps (up to eight images), the bank, pyramids and responses
    pairs = 8 * scales
    bound = pairs * (pixels * 184 + 8 * 55 * w * 8)
    bound += pairs * pixels * (4 + 36 + 4 + 4 + 4 + 72) + scales * pixels * 84 + 2 * 8 * pixels * 4
    assert used <= 1.1 * bound + (64 << 20), (used, bound)
    d.close()
