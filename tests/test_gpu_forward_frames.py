"""Forward projection along directions that are not finite, or point far beyond
the volume: their pixels read table entry 0, as the reference's clamped lookup
does, in the checked gather as in the unchecked one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf, 1e30, -3e9])
def test_bad_directions(cuda, oracle, ker32, bad, dtype):
    import torch

    from multigpugridder_amd import ops
    from multigpugridder_amd.synth import random_directions

    n = 16
    print(f"forward, direction component {bad}, {dtype}", flush=True)
    m, v = 2 * n, 2 * n + 6
    good = random_directions(12, 3).reshape(12, 9).astype(np.float32)
    axes = good.copy()
    for k in range(6):  # one component of u or v; frames 6 to 11 stay
        axes[k, k] = bad
    vol = torch.from_numpy(np.random.default_rng(4).uniform(1.0, 2.0, (v, v, v)).astype(np.float32)).to(cuda)
    vol = vol.to(getattr(torch, dtype))
    ker = torch.from_numpy(ker32).to(cuda)
    got, plain, ref = (ops.forward_project(vol, torch.from_numpy(a).to(cuda), m, ker=ker, **kw).cpu().numpy()
                       for a, kw in ((axes, {}), (axes, {"check": False}), (good, {})))
    assert np.array_equal(got[6:], ref[6:])
    if abs(bad) <= 1e30:  # the pixels at 0 along the bad component stay where they are
        want = oracle.forward_project(vol.float().cpu().numpy(), axes[:6], ker32, m)
        assert np.count_nonzero(want) > 0
        tol = 1e-5 * np.abs(want).max()  # FP32 sums of 64 products of one sign
        assert np.abs(got[:6] - want).max() <= tol and np.abs(plain[:6] - want).max() <= tol
    else:
        assert not got[:6].any() and not plain[:6].any()


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_bad_directions_generic_table(cuda, oracle, bad):
    """A table too large for the tile kernel takes the kernel of one pixel per thread."""
    import torch

    from multigpugridder_amd import ops
    from multigpugridder_amd.synth import random_directions

    n = 16
    print(f"forward, direction component {bad}, table 1001", flush=True)
    m, v = 2 * n, 2 * n + 6
    axes = random_directions(12, 3).reshape(12, 9).astype(np.float32)
    for k in range(6):
        axes[k, k] = bad
    vol = np.random.default_rng(4).uniform(1.0, 2.0, (v, v, v)).astype(np.float32)
    ker = oracle.kb_table(2, 1001).astype(np.float32)
    got = ops.forward_project(torch.from_numpy(vol).to(cuda), torch.from_numpy(axes).to(cuda), m,
                              ker=torch.from_numpy(ker).to(cuda)).cpu().numpy()
    assert not got[:6].any()
    want = oracle.forward_project(vol, axes[6:], ker, m)
    assert np.abs(got[6:] - want).max() <= 1e-5 * np.abs(want).max()
