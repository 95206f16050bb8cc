"""cas_images_to_images into memory that its input also lies in, reached through
another storage (as tensors imported from other libraries are)."""
import pytest
import torch


def test_overlap_is_by_address():
    from multigpugridder_amd import ops

    t = torch.zeros(100)
    part = torch.from_dlpack(t[60:])  # a storage of its own over the same memory
    assert part.untyped_storage().data_ptr() != t.untyped_storage().data_ptr()
    assert ops._overlap(t, part) and ops._overlap(part, t)
    assert not ops._overlap(t[:60], part)
    assert not ops._overlap(t[60:60], part)


@pytest.mark.gpu
def test_output_over_later_input(cuda):
    """More images than one pass of the chain takes: the first pass's output lies
    where the second reads."""
    from multigpugridder_amd import ops

    n, m, p = 16, 32, 600
    print(f"overlapping chain n={n} m={m} p={p}", flush=True)
    g = torch.Generator(device=cuda)
    g.manual_seed(6)
    cas = torch.randn((p, m, m), device=cuda, generator=g)
    want = ops.cas_images_to_images(cas, n)
    out = torch.from_dlpack(cas[450:]).view(p, n, n)
    assert torch.equal(ops.cas_images_to_images(cas, n, out=out), want)
