"""Stage calls captured into a caller's graph (torch.cuda.graph): the scratch that a captured
call names outlives larger calls and blink_release_cache, whoever allocates next.

Gridded cells are held to the bound of an FP32 sum (gridding_bounds), images to 1e-5 of the
peak of the FP64 image.
"""
import numpy as np
import pytest

import oracle
from gridding_bounds import assert_within, footprint_sums
from imager_amd import synth

pytestmark = pytest.mark.gpu

N = 64


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _images(g, c):
    want = np.fft.fftshift(np.fft.ifft2(g, norm="forward"), axes=(-2, -1))
    return want / c.sum(axis=(-2, -1))[:, None, None]


@pytest.mark.parametrize("K", [0, 5])
def test_captured_stage_calls_after_larger_ones(K):
    """Capture on scratch that is there (the slabs), then a larger call, a release of the cache
    and other allocations before the replays."""
    import torch
    from imager_amd import capi
    o = synth.small(n_ant=200, n_ch=40, n_t=1, n_pixels=N, seed=11 + K)
    d = [_dev(a) for a in (o.vis, o.u, o.v, o.flags, o.freq)]
    ref, cref, _ = oracle.gridding(o.vis, o.n_ant, o.u, o.v, o.flags, o.freq, o.delta_u, o.delta_v,
                                   o.min_uv, N, "XX", precision="f64", kernel_size=K, with_sinc=True)
    terms, sums = footprint_sums(o, N, K, True, o.vis[0, :, :, 0])

    def buffers(n_ch):
        return (torch.zeros((n_ch, N, N), dtype=torch.complex64, device="cuda"),
                torch.zeros((n_ch, N, N), device="cuda"),
                torch.empty((n_ch, N, N), dtype=torch.complex64, device="cuda"))

    def call(ctx, n_ch, grids, counts, images):
        args = (d[0], o.n_ant, n_ch, 1, d[1], d[2], d[3], d[4], o.delta_u, o.delta_v, o.min_uv, N, "XX", 0)
        if K:
            ctx.gridding_kernel(*args, K, grids, counts)
        else:
            ctx.gridding(*args, grids, counts)
        ctx.image(grids, counts, N, n_ch, images, zero_grids=False)

    def check(n_ch, grids, counts, images):
        torch.cuda.synchronize()
        assert np.array_equal(counts.cpu().numpy(), cref[0, :n_ch])
        assert_within(grids.cpu().numpy(), ref[0, :n_ch], terms[:n_ch], sums[:n_ch])
        want = _images(ref[0, :n_ch], cref[0, :n_ch])
        err = np.abs(images.cpu().numpy() - want).max(axis=(1, 2)) / np.abs(want).max(axis=(1, 2))
        assert err.max() < 1e-5

    with capi.Context() as ctx:
        small, large = buffers(8), buffers(40)
        print(f"K={K}: eager, 8 channels", flush=True)
        call(ctx, 8, *small)
        check(8, *small)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            call(ctx, 8, *small)
        print("larger call, release", flush=True)
        call(ctx, 40, *large)
        check(40, *large)
        ctx.release_cache()
        for t in large:
            t.zero_()
        call(ctx, 40, *large)
        check(40, *large)
        others = [torch.full((1 << k,), 7, dtype=torch.int32, device="cuda") for k in range(12, 24)]
        for replay in range(3):
            print("replay", replay, flush=True)
            for t in small:
                t.zero_()
            graph.replay()
            check(8, *small)
        assert all(int((t != 7).sum()) == 0 for t in others)
        del graph


@pytest.mark.parametrize("K", [0, 5])
def test_capture_without_scratch(K):
    """A capture that would have to allocate the cells of its channels holds the atomics."""
    import torch
    from imager_amd import capi
    o = synth.small(n_ant=200, n_ch=8, n_t=1, n_pixels=N, seed=23 + K)
    d = [_dev(a) for a in (o.vis, o.u, o.v, o.flags, o.freq)]
    ref, cref, _ = oracle.gridding(o.vis, o.n_ant, o.u, o.v, o.flags, o.freq, o.delta_u, o.delta_v,
                                   o.min_uv, N, "XX", precision="f64", kernel_size=K, with_sinc=True)
    terms, sums = footprint_sums(o, N, K, True, o.vis[0, :, :, 0])
    grids = torch.zeros((8, N, N), dtype=torch.complex64, device="cuda")
    counts = torch.zeros((8, N, N), device="cuda")

    def call(ctx, n_ch):
        args = (d[0], o.n_ant, n_ch, 1, d[1], d[2], d[3], d[4], o.delta_u, o.delta_v, o.min_uv, N, "XX", 0)
        if K:
            ctx.gridding_kernel(*args, K, grids, counts)
        else:
            ctx.gridding(*args, grids, counts)

    with capi.Context() as ctx:
        call(ctx, 1)                  # the kernel table, and cells for one channel at most
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            call(ctx, 8)
        for replay in range(4):
            grids.zero_()
            counts.zero_()
            if replay < 3:
                graph.replay()
            else:
                call(ctx, 8)          # eager: allocates, and takes the slabs
            torch.cuda.synchronize()
            assert np.array_equal(counts.cpu().numpy(), cref[0])
            assert_within(grids.cpu().numpy(), ref[0], terms, sums)
        del graph


def test_captured_images_of_a_small_side():
    """A capture of thousands of images of a small side, after images of an ordinary side
    only: the scratch does not grow with the call."""
    import torch
    from imager_amd import capi
    n, batch = 64, 4000
    gen = torch.Generator(device="cuda").manual_seed(1)
    grids = torch.view_as_complex(torch.randn((batch, n, n, 2), device="cuda", generator=gen))
    counts = torch.randint(1, 4, (batch, n, n), device="cuda", generator=gen).float()
    images = torch.empty_like(grids)
    want = torch.fft.fftshift(torch.fft.ifft2(grids.to(torch.complex128), norm="forward"), dim=(1, 2))
    want /= counts.double().sum(dim=(1, 2))[:, None, None]
    with capi.Context() as ctx:
        ordinary = torch.ones((1, 128, 128), dtype=torch.complex64, device="cuda")
        ctx.image(ordinary, torch.ones((1, 128, 128), device="cuda"), 128, 1, torch.empty_like(ordinary))
        torch.cuda.synchronize()
        # (the table of a side that blink_create does not prepare)
        ctx.fft2d_c2c(grids[:1], images[:1], n, 1)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            ctx.image(grids, counts, n, batch, images, zero_grids=False)
        for replay in range(3):
            images.zero_()
            graph.replay()
            torch.cuda.synchronize()
            err = (images - want).abs().amax(dim=(1, 2)) / want.abs().amax(dim=(1, 2))
            assert float(err.max()) < 1e-5
        del graph
