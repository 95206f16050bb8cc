"""Forward projection's bands and tiles per wave at direction counts around their
lines: every image as it comes out of a launch of its own (a tile's arithmetic
does not depend on the launch that it is in)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# bands of 8, 4, 2 and 1; 1, 2, 3 and 4 tiles per wave, checked and unchecked
@pytest.mark.parametrize("n,p", [(24, 31), (24, 100), (24, 128), (24, 255), (24, 257), (64, 33), (96, 17), (60, 90)])
@pytest.mark.parametrize("check", [None, False])
def test_same_as_alone(cuda, ker32, n, p, check):
    import torch

    from multigpugridder_amd import ops
    from multigpugridder_amd.synth import random_directions

    print(f"bands n={n} p={p} check={check}", flush=True)
    m, v = 2 * n, 2 * n + 6
    g = torch.Generator(device=cuda)
    g.manual_seed(n)
    vol = torch.randn((v, v, v), device=cuda, generator=g)
    axes = torch.from_numpy(np.ascontiguousarray(random_directions(p, 5).reshape(p, 9), dtype=np.float32)).to(cuda)
    ker = torch.from_numpy(ker32).to(cuda)
    out = torch.full((p, m, m), float("nan"), device=cuda)
    ops.forward_project(vol, axes, m, ker=ker, out=out, check=check)
    for a in list(range(0, p, max(1, p // 12))) + [p - 1]:
        assert torch.equal(out[a], ops.forward_project(vol, axes[a:a + 1], m, ker=ker, check=check)[0]), a
