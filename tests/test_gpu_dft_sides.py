"""The split-precision DFT transforms at the edges of their tiles: sides whose
half N/2 + 1 falls just below, on and just above a multiple of the 16 columns
of a step and the 32 rows of a matrix tile, the smallest sides (whose octets
do not fit the row) and the largest, with image counts that leave data tiles
partly filled.  Reference: the oracle's FP32 grid, transformed in float64."""
import numpy as np
import pytest

import oracle
from imager_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import torch
    from imager_amd import capi
    assert torch.cuda.is_available()
    return capi.Context()


@pytest.mark.parametrize("prec", ["BF16X3", "FP16X3"])
@pytest.mark.parametrize("n", [2, 4, 14, 16, 28, 30, 32, 34, 60, 62, 64, 66, 94, 126, 128, 190,
                               192, 254, 318, 478, 510, 512])
def test_dft_sides(ctx, prec, n):
    import torch
    from imager_amd import capi
    o = synth.small(n_ant=14, n_ch=3, n_t=1 if n % 4 else 2, n_pixels=n, seed=70 + n)
    grids, counts, _ = oracle.gridding(o.vis, o.n_ant, o.u, o.v, o.flags, o.freq, o.delta_u,
                                       o.delta_v, o.min_uv, n, "XX")
    g = np.asarray(grids).reshape(-1, n, n).astype(np.complex128)
    c = np.asarray(counts).reshape(-1, n * n).astype(np.float64).sum(1)
    ref = np.fft.fftshift(np.fft.ifft2(g), axes=(1, 2)).real * n * n / c[:, None, None]
    d = {k: torch.from_numpy(np.ascontiguousarray(getattr(o, k))).cuda()
         for k in ("vis", "u", "v", "w", "flags", "freq", "cable")}
    imgs = torch.full((o.n_images, n, n), float("nan"), dtype=torch.complex64, device="cuda")
    sums = torch.empty(o.n_images, dtype=torch.float64, device="cuda")
    st = capi.make_set(d["vis"], o.n_ant, o.n_ch, o.n_t, d["u"], d["v"], d["w"], d["flags"],
                       d["freq"], d["cable"], 0, o.delta_u, o.delta_v, o.min_uv, n, "XX", imgs,
                       sums, transform=getattr(capi, "TRANSFORM_DFT_" + prec))
    print("dft", prec, n, flush=True)
    ctx.image_batch([st])
    got = imgs.cpu().numpy()
    assert np.array_equal(sums.cpu().numpy(), c)
    assert np.all(got.imag == 0)
    # Per term and stage: both operands' splits and the dropped lo * lo are
    # 2^-18 (bf16) or 2^-24 (fp16) of the product each, and the folded sum and
    # difference of a pair double its terms: 3 x 2 x 2 stages.  FP32 sums of
    # 3 x 2 products per column: 6 K roundings at most per stage.  All of the
    # sum of |cells| over the count.
    unit = 2.0 ** (-18 if prec == "BF16X3" else -24)
    bound = (12 * unit + 12 * (n // 2 + 1) * 2.0 ** -24) * np.abs(g).sum((1, 2)) / c
    assert np.all(np.abs(got.real - ref).max((1, 2)) <= bound)
