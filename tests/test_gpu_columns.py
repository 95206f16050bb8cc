"""Back projection and the exact transpose by voxel columns, at the sizes where
their launchers choose them, against the oracle (or the tile scatter, which is
pinned to it)."""
import numpy as np
import pytest

from conftest import assert_parity

pytestmark = pytest.mark.gpu


def _frames(p, seed, skew=False):
    """Random rotations and, among them, axis permutations (all coordinates on
    the grid), 45 and 30 degree turns (table indices that are exactly
    half-integers), normals on the cube's diagonal, and left-handed frames."""
    from multigpugridder_amd.synth import random_directions

    axes = random_directions(p, seed).reshape(p, 3, 3).astype(np.float64)
    h, t = np.sqrt(0.5), np.sqrt(1 / 3)
    special = [np.roll(np.eye(3), k, axis=1) for k in range(3)]
    special += [np.array([[h, h, 0], [-h, h, 0], [0, 0, 1]]), np.array([[np.sqrt(0.75), 0.5, 0], [-0.5, np.sqrt(0.75), 0], [0, 0, 1]]),
                np.array([[1, 0, 0], [0, h, h], [0, -h, h]]), np.array([[0.5, 0, np.sqrt(0.75)], [0, 1, 0], [-np.sqrt(0.75), 0, 0.5]]),
                np.array([[h, -h, 0], [t * h, t * h, -2 * t * h], [t, t, t]]), np.diag([1.0, 1.0, -1.0])]
    axes[:len(special)] = special
    if skew:  # not orthonormal: the other kernel's share
        axes[20] *= 1.01
        axes[33, 1] += 0.05 * axes[33, 0]
        axes[34, 2] *= 0.99
    return np.ascontiguousarray(axes.reshape(p, 9), dtype=np.float32)


# V = 22 (one block deep, eight waves), 38, 66 (blocks hang over the edge);
# the shortest stack that takes columns, and a ragged one.
@pytest.mark.parametrize("n,p,mask,skew", [(8, 256, None, False), (16, 256, None, True), (16, 301, 9.0, False),
                                           (30, 259, None, True)])
def test_back_project(cuda, oracle, ker32, n, p, mask, skew):
    import torch

    from multigpugridder_amd import ops

    print(f"columns n={n} p={p} mask={mask} skew={skew}", flush=True)
    m, v = 2 * n, 2 * n + 6
    axes = _frames(p, 5, skew)
    imgs = np.random.default_rng(1).standard_normal((p, m, m)).astype(np.float32)
    start = np.random.default_rng(2).standard_normal((v, v, v)).astype(np.float32)
    out = torch.from_numpy(start).to(cuda)
    ops.back_project(torch.from_numpy(imgs).to(cuda), torch.from_numpy(axes).to(cuda), v, mask_radius=mask,
                     ker=torch.from_numpy(ker32).to(cuda), out=out)
    ref = oracle.back_project(imgs, axes, ker32, v, mask_radius=mask)
    assert_parity(out.cpu().numpy(), ref + start)


def test_back_project_four_waves(cuda, oracle, ker32):
    """V > 160: the four-wave kernel, 256 directions."""
    import torch

    from multigpugridder_amd import ops

    n, p = 80, 256
    print(f"columns n={n} p={p}", flush=True)
    m, v = 2 * n, 2 * n + 6
    axes = _frames(p, 6)
    imgs = np.random.default_rng(1).standard_normal((p, m, m)).astype(np.float32)
    got = ops.back_project(torch.from_numpy(imgs).to(cuda), torch.from_numpy(axes).to(cuda), v,
                           ker=torch.from_numpy(ker32).to(cuda))
    assert_parity(got.cpu().numpy(), oracle.back_project(imgs, axes, ker32, v))


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_non_finite_pixels_reach_the_windows_that_hold_them(cuda, ker32, bad):
    """A non-finite pixel anywhere leaves the whole call to the kernel that
    gathers all 25 taps (the same call without scratch)."""
    import torch

    from multigpugridder_amd import _lib, ops

    n, p = 16, 256
    m, v = 2 * n, 2 * n + 6
    imgs = torch.randn((p, m, m), device=cuda)
    imgs[3, 11, 17] = float(bad)
    axes, ker = torch.from_numpy(_frames(p, 5)).to(cuda), torch.from_numpy(ker32).to(cuda)
    got = ops.back_project(imgs, axes, v, ker=ker)
    ref = torch.zeros_like(got)
    _lib.call("mgg_op_back_project", ops._ptr(ref), None, v, ops._ptr(axes), p, ops._ptr(imgs), m, float(m / 2 - 1),
              ops._ptr(ker), 501, 2.0, ops._stream())
    assert not torch.isfinite(ref).all()
    assert torch.equal(torch.isnan(got), torch.isnan(ref))
    assert torch.equal(torch.nan_to_num(got), torch.nan_to_num(ref))


# V = 198 from 800 directions, V = 262 from 256; skewed frames go to the tiles.
@pytest.mark.parametrize("n,p,mask,skew", [(96, 800, None, True), (128, 256, 100.0, False)])
def test_transpose(cuda, ker32, n, p, mask, skew):
    import torch

    from multigpugridder_amd import ops

    print(f"transposed columns n={n} p={p} mask={mask} skew={skew}", flush=True)
    m, v = 2 * n, 2 * n + 6
    axes, ker = torch.from_numpy(_frames(p, 7, skew)).to(cuda), torch.from_numpy(ker32).to(cuda)
    imgs = torch.randn((p, m, m), device=cuda)
    for check in (None, ops.check_images(imgs, ker)):
        got = ops.back_project_adjoint(imgs, axes, v, mask_radius=mask, ker=ker, check=check)
        ref = ops.back_project_adjoint(imgs, axes, v, mask_radius=mask, ker=ker, check=False)
        assert_parity(got.cpu().numpy(), ref.cpu().numpy())
        # the columns gather in a fixed order
        if not skew:
            assert torch.equal(got, ops.back_project_adjoint(imgs, axes, v, mask_radius=mask, ker=ker))
