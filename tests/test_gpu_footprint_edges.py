"""Kaiser-Bessel footprints that reach the far edge of the plane.

calc_xy_grid2 (src/pacer_imager.cpp:716-750) keeps a footprint coordinate of -N, at
cell 0, and drops +N: there only one of a visibility's two footprints has the cell, and
the grid is not Hermitian.  Cells come that far when the oversampling times the
wavelength is under a metre or so (cells reach N / (oversampling * wavelength)).
"""
import numpy as np
import pytest

import oracle
from gridding_bounds import assert_within, footprint_sums, undersampled

pytestmark = pytest.mark.gpu


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


# (the sets of 24 and 10 antennas are sparse enough for the atomics, the others take the slabs)
@pytest.mark.parametrize("n_ant,n_ch,n,K", [(96, 2, 64, 7), (64, 2, 64, 12), (96, 3, 180, 8), (128, 5, 16, 7),
                                            (96, 2, 45, 7), (64, 2, 10, 9), (64, 2, 10, 10), (64, 3, 128, 5),
                                            (24, 1, 64, 7), (10, 1, 256, 9)])
def test_stage_footprints_at_the_far_edge(ctx, n_ant, n_ch, n, K):
    """blink_gridding_kernel on an undersampled plane, added to what is there."""
    import torch
    o = undersampled(n_ant, n_ch, n, seed=n_ant + n + K)
    d = [_dev(a) for a in (o.vis, o.u, o.v, o.flags, o.freq)]
    ref, cref, _ = oracle.gridding(o.vis, o.n_ant, o.u, o.v, o.flags, o.freq, 1.0, 1.0, o.min_uv,
                                   n, "XX", precision="f64", kernel_size=K, with_sinc=True)
    gen = torch.Generator(device="cuda").manual_seed(n)
    start = torch.randn((n_ch, n, n, 2), device="cuda", generator=gen)
    grids = torch.view_as_complex(start.clone())
    counts = torch.full((n_ch, n, n), 3.0, device="cuda")
    print(f"footprints at the far edge: {n_ant} antennas, {n_ch} x {n}^2, K={K}", flush=True)
    ctx.gridding_kernel(d[0], o.n_ant, n_ch, 1, d[1], d[2], d[3], d[4], 1.0, 1.0, o.min_uv, n,
                        "XX", 0, K, grids, counts)
    torch.cuda.synchronize()
    assert np.array_equal(counts.cpu().numpy(), 3.0 + cref[0])
    terms, sums = footprint_sums(o, n, K, True, o.vis[0, :, :, 0])
    s0 = torch.view_as_complex(start.double()).cpu().numpy()
    assert_within(grids.cpu().numpy(), s0 + ref[0], terms + 1.0, sums + np.abs(s0))


@pytest.mark.parametrize("n_ant,n_ch,n,K", [(96, 2, 64, 7), (64, 2, 64, 12), (96, 3, 180, 8), (128, 5, 16, 7),
                                            (64, 2, 10, 9), (64, 2, 10, 10), (40, 2, 16, 31), (64, 3, 256, 5),
                                            (24, 1, 512, 9), (160, 1, 14, 14)])
def test_batched_footprints_at_the_far_edge(ctx, n_ant, n_ch, n, K):
    """blink_image_batch on an undersampled plane: the real part of the image of the FP64
    grid, within the 1e-5 of the peak that every image is held to."""
    import torch
    from imager_amd import capi
    o = undersampled(n_ant, n_ch, n, seed=n_ant + n + K)
    d = [_dev(a) for a in (o.vis, o.u, o.v, o.w, o.flags, o.freq, o.cable)]
    g, c, _ = oracle.gridding(o.vis, o.n_ant, o.u, o.v, o.flags, o.freq, 1.0, 1.0, o.min_uv, n, "XX",
                              precision="f64", kernel_size=K, with_sinc=True)
    want = np.fft.fftshift(np.fft.ifft2(g[0], norm="forward"), axes=(-2, -1)).real
    want /= c[0].sum(axis=(-2, -1))[:, None, None]
    images = torch.full((1, n_ch, n, n), float("nan"), dtype=torch.complex64, device="cuda")
    sums = torch.empty(n_ch, dtype=torch.float64, device="cuda")
    print(f"batched footprints at the far edge: {n_ant} antennas, {n_ch} x {n}^2, K={K}", flush=True)
    ctx.image_batch([capi.make_set(d[0], o.n_ant, n_ch, 1, d[1], d[2], d[3], d[4], d[5], d[6], 0, 1.0,
                                   1.0, o.min_uv, n, "XX", images, sums, kernel_size=K)])
    torch.cuda.synchronize()
    assert np.array_equal(sums.cpu().numpy(), c[0].sum(axis=(-2, -1)))
    got = images.cpu().numpy()[0]
    assert (got.imag == 0).all()
    err = np.abs(got.real - want).max(axis=(-2, -1)) / np.abs(want).max(axis=(-2, -1))
    assert err.max() < 1e-5


@pytest.mark.parametrize("n", [7392, 7475, 7476, 8192])
def test_stage_footprints_around_the_largest_slab(ctx, n):
    """Sides around the largest whose row of cells and queues fit in LDS (7475), with a set
    dense enough for the slabs there."""
    import torch
    K = 31
    o = undersampled(72, 1, n, seed=n, reach=0.6)
    d = [_dev(a) for a in (o.vis, o.u, o.v, o.flags, o.freq)]
    ref, cref, _ = oracle.gridding(o.vis, o.n_ant, o.u, o.v, o.flags, o.freq, 1.0, 1.0, o.min_uv,
                                   n, "XX", precision="f64", kernel_size=K, with_sinc=True)
    grids = torch.zeros((1, n, n), dtype=torch.complex64, device="cuda")
    counts = torch.zeros((1, n, n), device="cuda")
    print(f"footprints around the largest slab: {n}^2", flush=True)
    ctx.gridding_kernel(d[0], o.n_ant, 1, 1, d[1], d[2], d[3], d[4], 1.0, 1.0, o.min_uv, n, "XX", 0,
                        K, grids, counts)
    torch.cuda.synchronize()
    assert np.array_equal(counts.cpu().numpy(), cref[0])
    terms, sums = footprint_sums(o, n, K, True, o.vis[0, :, :, 0])
    assert_within(grids.cpu().numpy(), ref[0], terms, sums)
