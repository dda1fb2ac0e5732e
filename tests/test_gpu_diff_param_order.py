"""A parameter change of the differentiation form against forwards still running on a stream
that the null stream does not wait for: each forward's responses equal those of a context created
with its parameters, bit for bit.
"""
import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu

PARAMS = [(0.56, 0.5), (0.61, 0.45), (0.5, 0.7)]


@pytest.fixture(scope="module")
def B():
    import bimp_amd
    if bimp_amd.device_count() < 1:
        pytest.fail("no GPU visible to the HIP library")
    return bimp_amd


@pytest.mark.parametrize("captured", [False, True])
def test_parameter_change_waits_for_the_forward(B, captured):
    import torch
    w, h, n, lam = 512, 512, 16, O.BASE_BANK
    img = np.stack([O.synth_frame(w, h, 12, i) for i in range(n)]).astype(np.float32)
    x = torch.from_numpy(img / np.float32(255)).cuda()
    d = B.Diff(w, h, lam)
    out = [torch.empty((n, d.response_size), device="cuda") for _ in range(3)]
    want = []
    for ratio, gamma in PARAMS:
        opt = B.default_options()
        opt.sigma_ratio, opt.gamma = ratio, gamma
        ref = B.Diff(w, h, lam, opt)
        r = torch.empty_like(out[0])
        ref.forward(x.data_ptr(), n, r.data_ptr())
        torch.cuda.synchronize()
        ref.close()
        want.append(r)
    side = torch.cuda.Stream()
    run = [lambda i=i: d.forward(x.data_ptr(), n, out[i].data_ptr(), side.cuda_stream)
           for i in range(3)]
    torch.cuda.synchronize()
    if captured:
        run[0]()
        side.synchronize()
        graphs = []
        for i in range(3):
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g, stream=side):
                run[i]()
            graphs.append(g)

        def replay(g):
            with torch.cuda.stream(side):
                g.replay()
        run = [lambda g=g: replay(g) for g in graphs]
    for _ in range(2):
        for i, (ratio, gamma) in enumerate(PARAMS):
            d.set_params(ratio, gamma)
            run[i]()
        side.synchronize()
        for i in range(3):
            assert torch.equal(out[i].view(torch.int32), want[i].view(torch.int32)), i
            out[i].zero_()
        torch.cuda.synchronize()
