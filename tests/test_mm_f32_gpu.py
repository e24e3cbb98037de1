"""mamba_mm_f32 (batched f32 products on f32 MFMA) over its tilings, layouts and
ragged edges, vs float64: a dot of k products of N(0, 1) values is off by at most
about k 2^-24 times the sum of their sizes, so 1e-5 sqrt(k) bounds it."""

import itertools

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# (z, m, n, k): one element, ragged 32-tiles, K over 4, 8 and 16 waves with
# ragged ends, odd rows (no 16-byte loads), 64-tiles with odd rows and with 16-byte
# loads up to ragged edges
SHAPES = [(1, 1, 1, 1), (3, 33, 31, 5), (2, 48, 250, 128), (2, 48, 250, 130),
          (2, 47, 251, 513), (1, 256, 100, 512), (5, 530, 515, 65), (4, 516, 508, 68)]


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


# both sides of the rows, channels and columns at which the block's out_proj moves
@pytest.mark.parametrize("rows,di,dm", [(1, 512, 256), (256, 512, 256), (257, 512, 256), (64, 528, 256), (64, 512, 264)])
def test_out_mm_on_both_sides_of_its_rule(rows, di, dm):
    import torch
    from mamba_hip.step import out_mm
    g = torch.Generator().manual_seed(rows + di)
    y, w = torch.randn(rows, di, generator=g), torch.randn(di, dm, generator=g)
    out = out_mm(y.cuda(), w.cuda())
    np.testing.assert_allclose(out.cpu().numpy(), (y.double() @ w.double()).numpy(), rtol=1e-4, atol=1e-5 * di ** 0.5)


def test_mamba1_block_on_both_sides_of_its_batch_rule(monkeypatch):
    """128 sequences on the own product, 129 on the library: the same rows."""
    import torch
    import mamba_hip
    from mamba_hip import mamba1
    calls = []
    own = mamba1.mm_f32
    monkeypatch.setattr(mamba1, "mm_f32", lambda *a: calls.append(1) or own(*a))
    m = mamba_hip.Mamba1Config(64).init("cuda", torch.Generator(device="cuda").manual_seed(2))
    x = torch.randn(129, 9, 64, generator=torch.Generator().manual_seed(3)).cuda()
    y, cache = m.forward(x[:128])
    assert calls
    n = len(calls)
    z, cache2 = m.forward(x)
    assert len(calls) == n
    torch.testing.assert_close(y, z[:128], rtol=1e-4, atol=1e-5)
    torch.testing.assert_close(cache.ssm_bir, cache2.ssm_bir[:128], rtol=1e-4, atol=1e-5)


def test_out_mm_under_autograd_and_forward_mode():
    import torch
    import torch.autograd.forward_ad as fw
    from mamba_hip.step import out_mm
    y, w, t = torch.randn(8, 64, device="cuda"), torch.randn(64, 32, device="cuda"), torch.randn(64, 32, device="cuda")
    with fw.dual_level():
        tangent = fw.unpack_dual(out_mm(y, fw.make_dual(w, t))).tangent
    torch.testing.assert_close(tangent, y @ t, rtol=1e-4, atol=1e-4)
    w.requires_grad_()
    out_mm(y, w).sum().backward()
    torch.testing.assert_close(w.grad, y.sum(0)[:, None].expand(64, 32), rtol=1e-4, atol=1e-4)
