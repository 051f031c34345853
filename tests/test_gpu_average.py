"""blink_image_averaging: image counts around its batches of 16, image sizes on both
sides of the size from which it takes the plain loop, and both forms.  The sum is
sequential FP32, exact to reproduce; the quotient may be off by one rounding."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,images", [(1, 1), (3, 2), (45, 16), (64, 17), (45, 18), (225, 32), (31, 33),
                                      (16, 768), (511, 20), (512, 1), (512, 19), (600, 3)])
@pytest.mark.parametrize("real_only", [False, True])
def test_average_is_the_sequential_mean(n, images, real_only):
    import torch
    from imager_amd import capi
    gen = torch.Generator(device="cuda").manual_seed(n + images)
    x = torch.randn((images, n, n, 2), device="cuda", generator=gen)
    want = x[0].clone()
    for k in range(1, images):
        want += x[k]
    want /= float(images)
    if real_only:
        want[..., 1] = 0.0
    out = torch.full((n, n), 7.0, dtype=torch.complex64, device="cuda")
    ctx = capi.Context()
    ctx.image_averaging(torch.view_as_complex(x), n * n, images, out, real_only)
    torch.cuda.synchronize()
    got = torch.view_as_real(out)
    assert bool(((got - want).abs() <= 2.0 ** -23 * want.abs()).all())
