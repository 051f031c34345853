"""The stage path's 2-D transform (blink_image, blink_fft2d_c2c) on grids that
gridding does not make: not Hermitian, with empty rows, cells that are -0.0,
counts where the grid is zero, several chunks of images.  Against torch's
FFT in complex128.

Tolerance: an FFT of length n = N^2 in FP32 has a relative 2-norm error of
at most about 5 u log2(n), u = 2^-24 (Higham, Accuracy and Stability of
Numerical Algorithms, sec. 24.1, twiddles rounded to FP32); a direct sum of a
prime radix R adds 2 R u per dimension.  The scale adds 2 u.
"""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def _tolerance(n):
    primes = sum(p for p in (7, 11, 13) if n % p == 0)
    return U * (5 * math.log2(n * n) + 4 * primes + 2)


def _shift(t, n):
    import torch
    h, odd = n // 2, n % 2
    p = np.arange(n)
    to = np.where(p < h, p + h + odd, p - h - odd)
    if odd:
        to[h] = h
    out = torch.empty_like(t)
    i = torch.from_numpy(to).cuda()
    out[:, i[:, None], i[None, :]] = t
    return out


def _grids(n, batch, seed):
    import torch
    gen = torch.Generator(device="cuda").manual_seed(seed)
    g = torch.zeros((batch, n, n, 2), dtype=torch.float32, device="cuda")
    g.normal_(generator=gen)
    g[:, n // 3:n // 2] = 0.0                       # empty rows
    g[:, :, ::3] = 0.0
    if n > 4:
        g[:, 1] = -0.0                              # a row of negative zeros
        g[0, 2] = 0.0
        g[0, 2, n - 1, 1] = 1.5                     # one component of one cell
    c = torch.randint(0, 4, (batch, n, n), device="cuda", generator=gen).float()
    return torch.view_as_complex(g), c


@pytest.mark.parametrize("n,batch", [(2, 3), (13, 2), (45, 3), (64, 5), (128, 3), (180, 2), (225, 3),
                                     (256, 3), (512, 3), (1001, 1), (1024, 25), (1500, 2), (2048, 2),
                                     (2002, 1), (4096, 2), (6000, 1)])
def test_image_of_any_grid(ctx, n, batch):
    import torch
    g, c = _grids(n, batch, seed=n)
    want = _shift(torch.fft.ifft2(g.to(torch.complex128), norm="forward") /
                  c.double().sum((1, 2))[:, None, None], n)
    for zero in (False, True):
        images = torch.full((batch, n, n), float("nan"), dtype=torch.complex64, device="cuda")
        gi, ci = g.clone(), c.clone()
        ctx.image(gi, ci, n, batch, images, zero_grids=zero)
        torch.cuda.synchronize()
        err = (torch.linalg.vector_norm(images.to(torch.complex128) - want) /
               torch.linalg.vector_norm(want)).item()
        print(f"image {n}^2 x {batch} zero={zero}: {err:.2e} of {_tolerance(n):.2e}", flush=True)
        assert err <= _tolerance(n)
        if zero:  # every bit cleared
            assert not torch.view_as_real(gi).view(torch.int32).any()
            assert not ci.view(torch.int32).any()
        else:
            assert torch.equal(torch.view_as_real(gi).view(torch.int32),
                               torch.view_as_real(g).view(torch.int32)) and torch.equal(ci, c)


@pytest.mark.parametrize("n,batch", [(2, 3), (90, 4), (128, 2), (256, 2), (512, 2), (1024, 22), (1125, 2),
                                     (2048, 1), (4096, 2)])
@pytest.mark.parametrize("direction", [1, -1])
def test_fft_in_place_and_out_of_place(ctx, n, batch, direction):
    import torch
    g, _ = _grids(n, batch, seed=n + direction)
    x = g.to(torch.complex128)
    want = torch.fft.ifft2(x, norm="forward") if direction > 0 else torch.fft.fft2(x)
    out = torch.full_like(g, float("nan"))
    ctx.fft2d_c2c(g, out, n, batch, direction)
    same = g.clone()
    ctx.fft2d_c2c(same, same, n, batch, direction)
    torch.cuda.synchronize()
    assert torch.equal(torch.view_as_real(out), torch.view_as_real(same))
    err = (torch.linalg.vector_norm(out.to(torch.complex128) - want) /
           torch.linalg.vector_norm(want)).item()
    print(f"fft {n}^2 x {batch} {direction}: {err:.2e} of {_tolerance(n):.2e}", flush=True)
    assert err <= _tolerance(n)


def test_image_nan_and_no_counts(ctx):
    """A NaN cell and counts of zero go where the arithmetic takes them: NaN images, cleared grids."""
    import torch
    g, c = _grids(256, 3, seed=4)
    g[0, 5, 7] = complex(float("nan"), 1.0)
    c[1] = 0.0
    images = torch.empty((3, 256, 256), dtype=torch.complex64, device="cuda")
    ctx.image(g, c, 256, 3, images)
    torch.cuda.synchronize()
    assert torch.isnan(images[0].real).all()
    assert not torch.isfinite(images[1].real).any()
    assert torch.isfinite(torch.view_as_real(images[2])).all()
    assert not torch.view_as_real(g).view(torch.int32).any()


@pytest.mark.parametrize("n", [3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 15, 16, 18, 26, 33, 36, 84, 96, 130, 192, 243, 400, 500, 729,
                               770, 968, 1040, 1331, 3072, 3125, 3600, 4004, 8192])
def test_every_radix(ctx, n):
    """Sides whose plans hold every radix, alone and together, one to four passes and more rows
    than a workgroup's threads hold at once, forward and backward."""
    import torch
    batch = 3 if n < 1000 else 1
    gen = torch.Generator(device="cuda").manual_seed(n)
    x = torch.view_as_complex(torch.randn((batch, n, n, 2), device="cuda", generator=gen))
    out = torch.empty_like(x)
    for direction, f in ((1, lambda t: torch.fft.ifft2(t, norm="forward")), (-1, torch.fft.fft2)):
        ctx.fft2d_c2c(x, out, n, batch, direction)
        torch.cuda.synchronize()
        want = f(x.to(torch.complex128))
        err = (torch.linalg.vector_norm(out.to(torch.complex128) - want) /
               torch.linalg.vector_norm(want)).item()
        print(f"fft {n}^2 {direction}: {err:.2e} of {_tolerance(n):.2e}", flush=True)
        assert err <= _tolerance(n)
