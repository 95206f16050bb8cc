"""Forward projection's order of the tiles and its one-index table rows: every
tile once, for direction and tile counts around the units the XCDs are dealt,
and weights for positions whose table index is exactly a half-integer."""
import numpy as np
import pytest

from conftest import assert_parity

pytestmark = pytest.mark.gpu


def _frames(p, seed):
    from multigpugridder_amd.synth import random_directions

    axes = random_directions(p, seed).reshape(p, 3, 3).astype(np.float64)
    h = np.sqrt(0.5)
    special = [np.eye(3), np.roll(np.eye(3), 1, axis=1), np.array([[np.sqrt(0.75), 0.5, 0], [-0.5, np.sqrt(0.75), 0], [0, 0, 1]]),
               np.array([[0.5, 0, np.sqrt(0.75)], [0, 1, 0], [-np.sqrt(0.75), 0, 0.5]]), np.array([[h, h, 0], [-h, h, 0], [0, 0, 1]])]
    n = min(p, len(special))
    axes[:n] = special[:n]
    return np.ascontiguousarray(axes.reshape(p, 9), dtype=np.float32)


# tiles per row: 1, 3, 5 (odd: half workgroup tiles), 8, 15; bands of an image
# below 64 directions, whole images from there, and counts that are no
# multiple of the 8 XCDs
@pytest.mark.parametrize("n,p", [(4, 1), (4, 65), (12, 7), (20, 1), (20, 9), (20, 63), (20, 64), (32, 3), (60, 2),
                                 (60, 33)])
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_every_tile(cuda, oracle, ker32, n, p, dtype):
    import torch

    from multigpugridder_amd import ops

    print(f"walk n={n} p={p} {dtype}", flush=True)
    m, v = 2 * n, 2 * n + 6
    axes = _frames(p, 3)
    cas = torch.from_numpy(np.random.default_rng(n).standard_normal((v, v, v)).astype(np.float32)).to(cuda)
    cas = cas.to(getattr(torch, dtype))
    out = torch.full((p, m, m), float("nan"), device=cuda)
    ops.forward_project(cas, torch.from_numpy(axes).to(cuda), m, ker=torch.from_numpy(ker32).to(cuda), out=out)
    assert_parity(out.cpu().numpy(), oracle.forward_project(cas.float().cpu().numpy(), axes, ker32, m))


def test_positions_below_one(cuda, oracle, ker32):
    """A mask that reaches past the volume's first voxels: windows that leave
    the volume, and positions where tap - position is rounded."""
    import torch

    from multigpugridder_amd import ops

    m, v, p = 40, 24, 12
    print(f"positions below one m={m} v={v}", flush=True)
    axes = _frames(p, 8)
    cas = np.random.default_rng(0).standard_normal((v, v, v)).astype(np.float32)
    got = ops.forward_project(torch.from_numpy(cas).to(cuda), torch.from_numpy(axes).to(cuda), m, mask_radius=19.0,
                              ker=torch.from_numpy(ker32).to(cuda))
    # the oracle, like the reference, bounds only the linear index; voxels
    # before the volume (negative index) are not read
    assert_parity(got.cpu().numpy(), oracle.forward_project(cas, axes, ker32, m, mask_radius=19.0))
