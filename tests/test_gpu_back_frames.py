"""Back projection along directions with a component that is not finite: all
their taps have weight 0, so they add nothing, whichever kernel meets them."""
import numpy as np
import pytest

from conftest import assert_parity

pytestmark = pytest.mark.gpu


# the bricks, with and without the density; the columns with the bad frames left
# to the bricks; a table of another size, which takes the generic kernel
@pytest.mark.parametrize("p,size,density", [(24, 501, False), (24, 501, True), (300, 501, False), (24, 301, True)])
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_bad_directions_add_nothing(cuda, oracle, bad, p, size, density):
    import torch

    from multigpugridder_amd import ops
    from multigpugridder_amd.synth import random_directions

    n = 16
    print(f"back, direction component {bad}, p={p}, table {size}, density {density}", flush=True)
    m, v = 2 * n, 2 * n + 6
    axes = random_directions(p, 3).reshape(p, 9).astype(np.float32)
    for k in range(9):
        axes[k, k] = bad
    imgs = np.random.default_rng(4).standard_normal((p, m, m)).astype(np.float32)
    ker = oracle.kb_table(2, size).astype(np.float32)
    got_den = torch.zeros((v, v, v), device=cuda) if density else None
    got = ops.back_project(torch.from_numpy(imgs).to(cuda), torch.from_numpy(axes).to(cuda), v,
                           ker=torch.from_numpy(ker).to(cuda), density=got_den)
    assert_parity(got.cpu().numpy(), oracle.back_project(imgs[9:], axes[9:], ker, v))
    if density:
        assert_parity(got_den.cpu().numpy(), oracle.back_project(np.ones_like(imgs[9:]), axes[9:], ker, v))
