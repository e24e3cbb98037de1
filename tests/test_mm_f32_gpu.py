"""mamba_mm_f32 (batched f32 products on f32 MFMA) over its tilings, layouts and
ragged edges, vs float64: a dot of k products of N(0, 1) values is off by at most
about k 2^-24 times the sum of their sizes, so 1e-5 sqrt(k) bounds it."""

import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# (z, m, n, k): one element, ragged 32-tiles, K over 4, 8 and 16 waves with
# ragged ends, odd rows (no 16-byte loads), 64-tiles
SHAPES = [(1, 1, 1, 1), (3, 33, 31, 5), (2, 48, 250, 128), (2, 48, 250, 130),
          (2, 47, 251, 513), (1, 256, 100, 512), (5, 530, 515, 65)]


@pytest.mark.parametrize("ta,tb", list(itertools.product([False, True], repeat=2)))
@pytest.mark.parametrize("shape", SHAPES)
def test_mm_f32(shape, ta, tb):
    import torch
    from mamba_hip.mamba1 import mm_f32
    z, m, n, k = shape
    g = torch.Generator().manual_seed(sum(shape))
    a = torch.randn((z, k, m) if ta else (z, m, k), generator=g)
    b = torch.randn((1, n, k) if tb else (1, k, n), generator=g)  # one matrix for the whole batch
    ad, bd = a.cuda(), b.cuda()
    out = mm_f32(ad.transpose(1, 2) if ta else ad, (bd.transpose(1, 2) if tb else bd).expand(z, -1, -1))
    torch.cuda.synchronize()
    want = (a.transpose(1, 2) if ta else a).double() @ (b.transpose(1, 2) if tb else b).double()
    np.testing.assert_allclose(out.cpu().numpy(), want.numpy(), rtol=1e-4, atol=1e-5 * k ** 0.5)


def test_mm_f32_refuses_operands_without_a_unit_stride():
    import torch
    import mamba_hip
    from mamba_hip.mamba1 import mm_f32
    a, b = torch.zeros(1, 4, 8, device="cuda")[:, ::2, ::2], torch.zeros(1, 4, 4, device="cuda")
    with pytest.raises(mamba_hip.MambaHipError):
        mm_f32(a, b)
