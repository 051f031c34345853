"""blink_image_batch over three output buffers in turn, without a wait between the calls: one
more than the graphs kept per call, so that every call re-points a graph whose
descriptor copy and replay may still be queued."""
import numpy as np
import pytest

import oracle
from imager_amd import synth

pytestmark = pytest.mark.gpu


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("n_sets", [3, 3000])
def test_rotating_buffers(n_sets):
    import torch
    from imager_amd import capi
    n = 16
    o = synth.small(n_ant=12, n_ch=1, n_t=1, n_pixels=n, seed=8)
    d = [_dev(a) for a in (o.vis, o.u, o.v, o.w, o.flags, o.freq, o.cable)]
    want, _ = oracle.run_f32(o.vis, o.n_ant, o.u, o.v, o.w, o.flags, o.freq, o.cable, True, True,
                             o.delta_u, o.delta_v, o.min_uv, n)
    want = want[0, 0].real
    out = [torch.full((n_sets, n, n), float("nan"), dtype=torch.complex64, device="cuda") for _ in range(3)]
    with capi.Context() as ctx:
        calls = [[capi.make_set(d[0], o.n_ant, 1, 1, d[1], d[2], d[3], d[4], d[5], d[6], 3, o.delta_u,
                                o.delta_v, o.min_uv, n, "XX", im) for im in images] for images in out]
        for k in range(12):
            ctx.image_batch(calls[k % 3])
        for images in out:
            images.fill_(float("nan"))
        for k in range(3):
            ctx.image_batch(calls[k])
        torch.cuda.synchronize()
    for images in out:
        got = images.cpu().numpy()
        assert np.abs(got.real - want).max() < 1e-5 * np.abs(want).max()
