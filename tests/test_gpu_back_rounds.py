"""Back projection of repeated directions: one group of gathered voxels then
names the same voxel once per copy, and every copy's contribution counts."""
import numpy as np
import pytest

from conftest import assert_parity

pytestmark = pytest.mark.gpu


# 1 and 2 copies, a pass of 128 directions filled with copies, and one beyond
# it; N = 4 puts many directions into one group.
@pytest.mark.parametrize("n,copies,density", [(4, 1, False), (4, 2, True), (4, 128, True), (16, 130, False)])
def test_repeated_directions_all_count(cuda, oracle, ker32, n, copies, density):
    import torch

    from multigpugridder_amd import ops
    from multigpugridder_amd.synth import random_directions

    print(f"back projection n={n} copies={copies} density={density}", flush=True)
    m, v = 2 * n, 2 * n + 6
    axes = np.repeat(random_directions(2, 9), copies, axis=0)
    imgs = np.random.default_rng(4).standard_normal((2 * copies, m, m)).astype(np.float32)
    den = torch.zeros((v, v, v), device=cuda) if density else None
    got = ops.back_project(torch.from_numpy(imgs).to(cuda), torch.from_numpy(axes).to(cuda), v,
                           ker=torch.from_numpy(ker32).to(cuda), density=den)
    assert_parity(got.cpu().numpy(), oracle.back_project(imgs, axes, ker32, v))
    if density:
        assert_parity(den.cpu().numpy(), oracle.back_project(np.ones_like(imgs), axes, ker32, v))
