"""More sets in one batched call than a launch has blocks along y or z (65535)."""
import numpy as np
import pytest

import oracle
from imager_amd import synth

pytestmark = pytest.mark.gpu


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("K,n,n_ant", [(3, 8, 4), (0, 2, 20)])
def test_batch_of_many_sets(K, n, n_ant):
    """65540 single-image sets, convolutional, and nearest-cell sets dense enough for the
    direct row pass: every image within 1e-5 of the peak of the oracle's."""
    import torch
    from imager_amd import capi
    o = synth.small(n_ant=n_ant, n_ch=1, n_t=1, n_pixels=n, seed=5)
    o.oversampling, (o.u_max, o.v_max, o.delta_u, o.delta_v) = 2.0, synth.grid_scalars(o.u, o.v, o.flags, n)
    n_sets = 65540
    d = [_dev(a) for a in (o.vis, o.u, o.v, o.w, o.flags, o.freq, o.cable)]
    images = torch.full((n_sets, n, n), float("nan"), dtype=torch.complex64, device="cuda")
    g, c, _ = oracle.gridding(o.vis, o.n_ant, o.u, o.v, o.flags, o.freq, o.delta_u, o.delta_v,
                              o.min_uv, n, "XX", kernel_size=K)
    want = oracle.image(g, c)[0, 0].real
    with capi.Context() as ctx:
        print(f"{n_sets} sets of {n}^2, K={K}", flush=True)
        sets = [capi.make_set(d[0], o.n_ant, 1, 1, d[1], d[2], d[3], d[4], d[5], d[6], 0, o.delta_u,
                              o.delta_v, o.min_uv, n, "XX", images[i], kernel_size=K)
                for i in range(n_sets)]
        ctx.image_batch(sets)
        torch.cuda.synchronize()
    got = images.cpu().numpy()
    assert (got.imag == 0).all()
    assert np.abs(got.real - want).max() < 1e-5 * np.abs(want).max()
