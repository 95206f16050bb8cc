"""Volume chains at the sizes of the fused passes (M = 128, 192, 256, 384, 512),
several N of each and paddings, against a float64 transform of the same volume
(the oracle's chain, by torch on the GPU where numpy would take long)."""
import numpy as np
import pytest

from conftest import rel_l2

pytestmark = pytest.mark.gpu

TOL = 1e-6  # an FP32 transform of 2^24..2^27 values: log2(M^3) roundings of 6e-8, in quadrature


def _shift(x):
    import torch
    return torch.fft.fftshift(x)


def _vol_to_cas(vol, oracle, m, pad):
    import torch
    n = vol.shape[0]
    pc = torch.from_numpy(oracle.precomp(m)).to(vol.device)
    x = torch.nn.functional.pad(vol.double(), ((m - n) // 2,) * 6) * pc[:, None, None] * pc[None, :, None] * pc
    f = _shift(torch.fft.fftn(_shift(x)))
    return torch.nn.functional.pad(f.real + f.imag, (pad,) * 6)


def _cas_to_vol(cas, oracle, m, pad, n, keep):
    import torch
    c = cas.double()[pad:pad + m, pad:pad + m, pad:pad + m]
    mir = torch.roll(torch.flip(c, (0, 1, 2)), (1, 1, 1), (0, 1, 2))
    z = torch.complex(0.5 * (c + mir), 0.5 * (c - mir))
    if not keep:
        z[0] = 0
        z[:, 0] = 0
        z[:, :, 0] = 0
    x = _shift(torch.fft.ifftn(_shift(z))).real
    pc = torch.from_numpy(oracle.precomp(m)).to(cas.device)
    x = x * pc[:, None, None] * pc[None, :, None] * pc
    o = (m - n) // 2
    return x[o:o + n, o:o + n, o:o + n]


# N = M / 2; small N (one workgroup's rows are several planes); N without a
# factor 8 (lines beyond the last XCD round); N = M - 2, the largest; no padding
@pytest.mark.parametrize("n,m,pad", [(64, 128, 3), (2, 128, 3), (126, 128, 0), (96, 192, 3), (50, 192, 5), (128, 256, 3),
                                     (64, 256, 1), (100, 256, 3), (192, 384, 3), (256, 512, 3), (130, 512, 0)])
def test_fused_volume_chains(cuda, oracle, n, m, pad):
    import torch

    from multigpugridder_amd import _lib, ops

    print(f"volume chains n={n} m={m} pad={pad}", flush=True)
    v = m + 2 * pad
    vol = torch.randn((n, n, n), device=cuda)
    cas = torch.full((v, v, v), float("nan"), device=cuda)
    _lib.call("mgg_op_volume_to_cas_volume", ops._ptr(vol), n, ops._ptr(cas), m, pad, 2.0, ops._stream())
    assert rel_l2(cas.cpu().numpy(), _vol_to_cas(vol, oracle, m, pad).cpu().numpy()) < TOL
    if pad:  # the padding is exactly zero
        inner = cas.clone()
        inner[pad:-pad, pad:-pad, pad:-pad] = 0
        assert not inner.any()
    noise = torch.randn((v, v, v), device=cuda)
    for keep in (False, True):
        out = torch.full((n, n, n), float("nan"), device=cuda)
        _lib.call("mgg_op_cas_volume_to_volume", ops._ptr(noise), m, pad, ops._ptr(out), n, 2.0, int(not keep),
                  ops._stream())
        assert rel_l2(out.cpu().numpy(), _cas_to_vol(noise, oracle, m, pad, n, keep).cpu().numpy()) < TOL
