"""The inverse image chain drops the index-0 row and column of its CAS images
whatever they hold, also at the sizes with kernels of their own, and on both
sides of the line between these and the general passes (M = 384 and 512)."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,m", [(64, 128), (128, 128), (96, 192), (128, 256), (240, 384), (242, 384), (320, 512),
                                 (322, 512)])
def test_images(cuda, n, m):
    import torch

    from multigpugridder_amd import ops

    print(f"index 0 of CAS images n={n} m={m}", flush=True)
    g = torch.Generator(device=cuda)
    g.manual_seed(5)
    imgs = torch.randn((3, m, m), device=cuda, generator=g)
    imgs[:, 0] = 0
    imgs[:, :, 0] = 0
    bad = imgs.clone()
    bad[:, 0] = float("nan")
    bad[:, :, 0] = float("inf")
    want = ops.cas_images_to_images(imgs, n)
    assert torch.isfinite(want).all()
    assert torch.equal(ops.cas_images_to_images(bad, n), want)
