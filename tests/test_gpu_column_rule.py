"""Back projection and the transpose at the sizes where the choice between the
columns and the bricks (or tiles), and of the waves per brick, changes: the call
with scratch against the one without, which keeps the bricks (pinned to the
oracle elsewhere)."""
import numpy as np
import pytest

from conftest import assert_parity

pytestmark = pytest.mark.gpu


# Shortest stacks that take columns, and the longest that do not, by the place of
# the volume's centre in a brick (V / 2 mod 8): V = 62 and 206 (7), 66 (1), 166 and
# 182 (3), 262 (3: the usual N = 128), 306 (1); V = 176 and 178 have eight and four waves.
@pytest.mark.parametrize("n,p", [(28, 1499), (28, 1500), (30, 799), (30, 801), (80, 499), (80, 500), (85, 500), (86, 800),
                                 (88, 256), (100, 1500), (128, 1000), (150, 500)])
def test_back_project(cuda, ker32, n, p):
    import torch

    from multigpugridder_amd import _lib, ops
    from multigpugridder_amd.synth import random_directions

    print(f"columns' lines n={n} p={p}", flush=True)
    m, v = 2 * n, 2 * n + 6
    g = torch.Generator(device=cuda)
    g.manual_seed(n)
    imgs = torch.randn((p, m, m), device=cuda, generator=g)
    axes = torch.from_numpy(np.ascontiguousarray(random_directions(p, 5).reshape(p, 9), dtype=np.float32)).to(cuda)
    ker = torch.from_numpy(ker32).to(cuda)
    got = ops.back_project(imgs, axes, v, ker=ker)
    ref = torch.zeros_like(got)
    _lib.call("mgg_op_back_project", ops._ptr(ref), None, v, ops._ptr(axes), p, ops._ptr(imgs), m, float(m / 2 - 1),
              ops._ptr(ker), 501, 2.0, ops._stream())
    # a wave adds the directions of a voxel one after the other, at most p / 4
    # in FP32; a flipped rounding decision is 1e-4 of the peak
    assert_parity(got.cpu().numpy(), ref.cpu().numpy(), peak=max(2e-6, p / 4 * 2.0 ** -24))
