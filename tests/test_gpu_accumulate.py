"""LDS accumulation of gridded visibilities where many fall on one cell.

The gridding kernels add complex values to LDS cells with a 64-bit
compare-and-swap; every lane of a wavefront on one cell is its worst case.
The FP32 sum of n values in any order lies within n 2^-24 sum |v| of the exact
sum.
"""
import numpy as np
import pytest

import oracle
from imager_amd import synth

pytestmark = pytest.mark.gpu


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _crowded(n_ant, n_pixels, cells, seed):
    """An observation whose unflagged baselines share `cells` uv positions."""
    o = synth.small(n_ant=n_ant, n_ch=1, n_t=1, n_pixels=n_pixels, seed=seed)
    rng = np.random.Generator(np.random.PCG64(seed))
    pick = rng.integers(0, cells, o.n_bl)
    pos = rng.uniform(-0.2, 0.2, (2, cells)) * n_pixels
    lam = synth.C_LIGHT / o.freq[0]
    o.delta_u = o.delta_v = 1.0
    o.u = (pos[0][pick] * lam).astype(np.float32)
    o.v = (pos[1][pick] * lam).astype(np.float32)
    return o


@pytest.mark.parametrize("n_ant,n,cells", [(40, 64, 1), (65, 180, 2), (128, 128, 3), (256, 256, 1)])
def test_crowded_cells(ctx, n_ant, n, cells):
    import torch
    from imager_amd import capi
    o = _crowded(n_ant, n, cells, seed=n_ant + cells)
    d = [_dev(a) for a in (o.vis, o.u, o.v, o.flags, o.freq)]
    ref, cref, _ = oracle.gridding(o.vis.astype(np.complex64), o.n_ant, o.u, o.v, o.flags, o.freq,
                                   1.0, 1.0, o.min_uv, n, "XX", precision="f64")
    n_bl = o.n_bl
    bound = n_bl * 2.0 ** -24 * np.abs(o.vis[0, 0, :, 0]).sum()
    for algo in (capi.GRID_TILED, capi.GRID_ATOMIC):
        grids = torch.zeros((1, 1, n, n), dtype=torch.complex64, device="cuda")
        counts = torch.zeros((1, 1, n, n), dtype=torch.float32, device="cuda")
        ctx.gridding(d[0], o.n_ant, 1, 1, d[1], d[2], d[3], d[4], 1.0, 1.0, o.min_uv, n, "XX", 0,
                     grids, counts, algo=algo)
        torch.cuda.synchronize()
        assert np.array_equal(counts.cpu().numpy(), cref)
        assert np.abs(grids.cpu().numpy() - ref).max() <= bound


@pytest.mark.parametrize("n,transform", [(128, 0), (180, 0), (256, 0), (180, 2)])
@pytest.mark.parametrize("direct", ["0", "1"])
def test_crowded_cells_batched(ctx, monkeypatch, n, transform, direct):
    import torch
    from imager_amd import capi
    monkeypatch.setenv("BLINK_DIRECT", direct)
    o = _crowded(96, n, 2, seed=n)
    d = [_dev(a) for a in (o.vis, o.u, o.v, o.w, o.flags, o.freq, o.cable)]
    images = torch.empty((1, 1, n, n), dtype=torch.complex64, device="cuda")
    ctx.image_batch([capi.make_set(d[0], o.n_ant, 1, 1, d[1], d[2], d[3], d[4], d[5], d[6], 3, 1.0,
                                   1.0, o.min_uv, n, "XX", images, transform=transform)])
    torch.cuda.synchronize()
    ref, _ = oracle.run_f32(o.vis, o.n_ant, o.u, o.v, o.w, o.flags, o.freq, o.cable, True, True,
                            1.0, 1.0, o.min_uv, n)
    assert oracle.peak_normalised_error(images.cpu().numpy(), ref)[0] < 1e-5


@pytest.mark.parametrize("n_ant,n_ch,n_t,n", [(96, 3, 2, 128), (256, 3, 1, 225), (128, 9, 1, 512), (64, 40, 1, 45),
                                              (256, 17, 1, 1024), (160, 1, 1, 2), (33, 300, 1, 16)])
@pytest.mark.parametrize("pol,min_uv", [("XX", -np.inf), ("V", 2.0)])
def test_stage_gridding_adds_to_what_is_there(ctx, n_ant, n_ch, n_t, n, pol, min_uv):
    """blink_gridding accumulates: twice over the same cells of non-empty grids, odd and even
    sides, both sides of the choice between slabs and atomics.  Counts exact; sums within the
    bound of an FP32 sum of the cell's values and what was there."""
    import torch
    from imager_amd import capi
    o = synth.small(n_ant=n_ant, n_ch=n_ch, n_t=n_t, n_pixels=n, seed=n_ant + n, bl_flag_fraction=0.2)
    o.vis[0, 0, 3, :] = np.nan
    d = [_dev(a) for a in (o.vis, o.u, o.v, o.flags, o.freq)]
    ref, cref, _ = oracle.gridding(o.vis, o.n_ant, o.u, o.v, o.flags, o.freq, o.delta_u, o.delta_v,
                                   min_uv, n, pol, precision="f64")
    gen = torch.Generator(device="cuda").manual_seed(n)
    start = torch.randn((n_t, n_ch, n, n, 2), device="cuda", generator=gen)
    grids = torch.view_as_complex(start.clone())
    counts = torch.full((n_t, n_ch, n, n), 5.0, device="cuda")
    for _ in range(2):
        ctx.gridding(d[0], o.n_ant, n_ch, n_t, d[1], d[2], d[3], d[4], o.delta_u, o.delta_v, min_uv, n,
                     pol, 0, grids, counts)
    torch.cuda.synchronize()
    assert np.array_equal(counts.cpu().numpy(), 5.0 + 2.0 * cref)
    want = torch.view_as_complex(start.double()).cpu().numpy() + 2.0 * ref
    big = float(np.nanmax(np.abs(o.vis))) * 2.0
    terms = 2.0 * cref.max() + 2.0
    assert np.abs(grids.cpu().numpy() - want).max() <= terms * 2.0 ** -24 * (terms * big + 10.0)


@pytest.mark.parametrize("n_ant,n_ch,n,K", [(48, 2, 64, 1), (40, 3, 45, 7), (64, 1, 180, 8), (64, 2, 225, 9),
                                            (96, 5, 256, 7), (24, 1, 16, 31), (200, 1, 61, 16), (10, 1, 1024, 7),
                                            (128, 2, 1001, 4), (32, 2, 10, 9), (32, 2, 10, 10), (32, 1, 8, 9)])
@pytest.mark.parametrize("pol,min_uv", [("XX", -np.inf), ("I", 2.0)])
def test_stage_footprints_add_to_what_is_there(ctx, n_ant, n_ch, n, K, pol, min_uv):
    """blink_gridding_kernel over its slabs and its atomics (the smallest and sparsest sets), odd and
    even sides and footprints, footprints wider than a slab or cut by the plane's edge, twice
    over non-empty grids.  Counts exact; sums within the bound of an FP32 sum."""
    import torch
    o = synth.small(n_ant=n_ant, n_ch=n_ch, n_t=1, n_pixels=n, seed=n_ant + n + K, bl_flag_fraction=0.2)
    o.vis[0, 0, 5, :] = np.nan
    d = [_dev(a) for a in (o.vis, o.u, o.v, o.flags, o.freq)]
    ref, cref, _ = oracle.gridding(o.vis, o.n_ant, o.u, o.v, o.flags, o.freq, o.delta_u, o.delta_v,
                                   min_uv, n, pol, precision="f64", kernel_size=K, with_sinc=True)
    gen = torch.Generator(device="cuda").manual_seed(n)
    start = torch.randn((1, n_ch, n, n, 2), device="cuda", generator=gen)
    grids = torch.view_as_complex(start.clone())
    counts = torch.full((1, n_ch, n, n), 3.0, device="cuda")
    for _ in range(2):
        ctx.gridding_kernel(d[0], o.n_ant, n_ch, 1, d[1], d[2], d[3], d[4], o.delta_u, o.delta_v,
                            min_uv, n, pol, 0, K, grids, counts)
    torch.cuda.synchronize()
    assert np.array_equal(counts.cpu().numpy(), 3.0 + 2.0 * cref)
    want = torch.view_as_complex(start.double()).cpu().numpy() + 2.0 * ref
    weight = float(np.abs(oracle.kb_kernels(K)).max()) ** 2
    big = float(np.nanmax(np.abs(o.vis))) * max(weight, 1.0)
    terms = 4.0 * o.n_bl
    assert np.abs(grids.cpu().numpy() - want).max() <= terms * 2.0 ** -24 * (big + 10.0)


@pytest.mark.parametrize("n", [7392, 7488, 8192])
def test_stage_footprints_of_the_largest_sides(ctx, n):
    """Sides around the largest whose row of cells and queues fit in LDS (7475), with a set
    dense enough that slabs would pay on either.  Counts exact; sums within the bound of an FP32 sum."""
    import torch
    K = 31
    o = synth.small(n_ant=72, n_ch=1, n_t=1, n_pixels=n, seed=n)
    d = [_dev(a) for a in (o.vis, o.u, o.v, o.flags, o.freq)]
    ref, cref, _ = oracle.gridding(o.vis, o.n_ant, o.u, o.v, o.flags, o.freq, o.delta_u, o.delta_v,
                                   o.min_uv, n, "XX", precision="f64", kernel_size=K, with_sinc=True)
    grids = torch.zeros((1, 1, n, n), dtype=torch.complex64, device="cuda")
    counts = torch.zeros((1, 1, n, n), device="cuda")
    ctx.gridding_kernel(d[0], o.n_ant, 1, 1, d[1], d[2], d[3], d[4], o.delta_u, o.delta_v,
                        o.min_uv, n, "XX", 0, K, grids, counts)
    torch.cuda.synchronize()
    assert np.array_equal(counts.cpu().numpy(), cref)
    weight = float(np.abs(oracle.kb_kernels(K)).max()) ** 2
    big = float(np.abs(o.vis).max()) * max(weight, 1.0)
    # a cell sees the footprints of at most n_bl visibilities and their conjugates
    err = np.abs(grids.cpu().numpy() - ref).max()
    assert err <= 2.0 * o.n_bl * 2.0 ** -24 * 2.0 * o.n_bl * big


@pytest.mark.parametrize("K", [0, 5])
def test_stage_gridding_captured_without_scratch(K):
    """A capture that needs more scratch for the cells than the context holds takes the atomics;
    replays match the eager call.  Sums within the bound of two FP32 sums in different orders."""
    import torch
    from imager_amd import capi
    ctx = capi.Context()
    n, o = 64, synth.small(n_ant=64, n_ch=8, n_t=1, n_pixels=64, seed=3)
    d = [_dev(a) for a in (o.vis, o.u, o.v, o.flags, o.freq)]
    grids = torch.zeros((1, 8, n, n), dtype=torch.complex64, device="cuda")
    counts = torch.zeros((1, 8, n, n), device="cuda")

    def call(n_ch):
        args = (d[0], o.n_ant, n_ch, 1, d[1], d[2], d[3], d[4], o.delta_u, o.delta_v, o.min_uv, n, "XX", 0)
        if K:
            ctx.gridding_kernel(*args, K, grids, counts)
        else:
            ctx.gridding(*args, grids, counts)

    call(1)                       # the kernel table, and cells for one channel at most
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(8)
    got = []
    for _ in range(3):
        grids.zero_()
        counts.zero_()
        graph.replay()
        torch.cuda.synchronize()
        got.append((grids.cpu().numpy().copy(), counts.cpu().numpy().copy()))
    grids.zero_()
    counts.zero_()
    call(8)                       # eager: may allocate, and take the slabs
    torch.cuda.synchronize()
    big = float(np.abs(o.vis).max()) * (float(np.abs(oracle.kb_kernels(K)).max()) ** 2 if K else 1.0)
    for g, c in got:
        assert np.array_equal(c, counts.cpu().numpy())
        terms = 2.0 * o.n_bl
        assert np.abs(g - grids.cpu().numpy()).max() <= 2.0 * terms * 2.0 ** -24 * terms * big
