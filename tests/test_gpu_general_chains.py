"""Image and volume chains at even sizes without kernels of their own (any
factors 2, 3, 5, 7, 11, 13 up to 512) and at sizes left to rocFFT, against
float64 transforms of the same input."""
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

TOL = 1e-6  # an FP32 transform of at most 2^27 values: log2 roundings of 6e-8, in quadrature


def _fwd(x, m, dims):
    """Pad, shift, transform, shift, CAS; in float64."""
    import torch
    n = x.shape[-1]
    x = torch.nn.functional.pad(x.double(), ((m - n) // 2,) * (2 * len(dims)))
    f = torch.fft.fftshift(torch.fft.fftn(torch.fft.fftshift(x, dims), dim=dims), dims)
    return f.real + f.imag


def _inv(cas, n, dims, drop):
    import torch
    c = cas.double()
    m = c.shape[-1]
    mir = torch.roll(torch.flip(c, dims), (1,) * len(dims), dims)
    z = torch.complex(0.5 * (c + mir), 0.5 * (c - mir))
    if drop:
        for d in dims:
            z.select(d, 0).zero_()
    x = torch.fft.fftshift(torch.fft.ifftn(torch.fft.fftshift(z, dims), dim=dims), dims).real
    o = (m - n) // 2
    for d in dims:
        x = x.narrow(d, o, n)
    return x


# every radix alone and together, both sides of the rule of M = 384 and 512, the smallest sizes, one and two workgroups of
# lines, 8 transforms per workgroup, a batch beyond one scratch (image_batch),
# and rocFFT's (factor 17; 514)
@pytest.mark.parametrize("p,n,m", [(1, 2, 2), (3, 2, 6), (2, 8, 16), (5, 6, 22), (3, 14, 26), (3, 30, 30), (7, 50, 98),
                                   (300, 98, 100), (3, 50, 100), (2, 64, 128), (3, 154, 154), (2, 100, 250), (2, 128, 260), (2, 364, 364),
                                   (2, 242, 486), (2, 250, 500), (2, 2, 512), (2, 20, 34), (2, 256, 514),
                                   (2, 240, 384), (2, 242, 384), (2, 320, 512), (2, 322, 512)])
def test_image_chains(cuda, p, n, m):
    import torch

    from multigpugridder_amd import ops

    print(f"image chains p={p} n={n} m={m}", flush=True)
    imgs = torch.randn((p, n, n), device=cuda)
    got = ops.images_to_cas_images(imgs, m)
    want = _fwd(imgs, m, (1, 2))
    assert rel_l2(got.cpu().numpy(), want.cpu().numpy()) < TOL
    t = ops.cas_images_to_images_transpose(imgs, m)
    want = want / (m * m)
    want[:, 0] = 0
    want[:, :, 0] = 0
    assert rel_l2(t.cpu().numpy(), want.cpu().numpy()) < TOL

    cas = torch.randn((p, m, m), device=cuda)
    want = _inv(cas, n, (1, 2), True).cpu().numpy()
    keep = cas.clone()
    assert rel_l2(ops.cas_images_to_images(cas, n).cpu().numpy(), want) < TOL
    assert torch.equal(cas, keep)  # the caller's stack stays as it is
    # an output over the input's memory (the stack's own front)
    out = cas.view(-1)[:p * n * n].view(p, n, n)
    assert rel_l2(ops.cas_images_to_images(cas, n, out=out).cpu().numpy(), want) < TOL


@pytest.mark.parametrize("n,m,pad", [(2, 6, 3), (30, 78, 0), (40, 80, 3), (78, 80, 0), (30, 90, 1), (50, 100, 3), (98, 154, 3),
                                     (64, 130, 3), (120, 240, 3), (100, 300, 5), (150, 308, 0), (20, 34, 3)])
def test_volume_chains(cuda, oracle, n, m, pad):
    import torch

    from multigpugridder_amd import _lib, ops

    print(f"volume chains n={n} m={m} pad={pad}", flush=True)
    v = m + 2 * pad
    pc = torch.from_numpy(oracle.precomp(m)).to(cuda)
    o = (m - n) // 2
    w = (pc[:, None, None] * pc[None, :, None] * pc)[o:o + n, o:o + n, o:o + n]
    vol = torch.randn((n, n, n), device=cuda)
    cas = torch.full((v, v, v), float("nan"), device=cuda)
    _lib.call("mgg_op_volume_to_cas_volume", ops._ptr(vol), n, ops._ptr(cas), m, pad, 2.0, ops._stream())
    want = torch.nn.functional.pad(_fwd(vol.double() * w, m, (0, 1, 2)), (pad,) * 6)
    assert rel_l2(cas.cpu().numpy(), want.cpu().numpy()) < TOL
    noise = torch.randn((v, v, v), device=cuda)
    for keep in (True, False):
        out = torch.full((n, n, n), float("nan"), device=cuda)
        _lib.call("mgg_op_cas_volume_to_volume", ops._ptr(noise), m, pad, ops._ptr(out), n, 2.0, int(not keep),
                  ops._stream())
        want = _inv(noise[pad:pad + m, pad:pad + m, pad:pad + m], n, (0, 1, 2), not keep) * w
        assert rel_l2(out.cpu().numpy(), want.cpu().numpy()) < TOL


# The index-0 row, column and planes of the inverse chains are dropped whatever
# they hold: sizes with and without kernels of their own and rocFFT's.
@pytest.mark.parametrize("n,m", [(64, 128), (50, 100), (20, 34)])
def test_index_zero_is_dropped(cuda, n, m):
    import torch

    from multigpugridder_amd import ops

    vol = torch.randn((m + 6,) * 3, device=cuda)
    bad = vol.clone()
    bad[3] = float("nan")
    bad[:, 3] = float("inf")
    bad[:, :, 3] = float("nan")
    a, b = (ops.cas_volume_to_volume(x, n, interp_factor=m / n) for x in (vol, bad))
    assert torch.equal(a, b)
    if m == 128:  # its row kernel multiplies by zero
        return
    imgs = torch.randn((2, m, m), device=cuda)
    bad = imgs.clone()
    bad[:, 0] = float("nan")
    bad[:, :, 0] = float("inf")
    assert torch.equal(ops.cas_images_to_images(imgs, n), ops.cas_images_to_images(bad, n))
