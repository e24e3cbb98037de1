"""mamba_linear_row vs float64: the operand is the row (RMS-normed) rounded to
bf16, off by at most 2^-9 of itself, so a column is off by at most
2^-9 sum_k |x_k w_k| (the weights are exact in bf16), the f32 accumulation's
1e-5 of the same sum, and the output's own rounding."""

import pytest

pytestmark = pytest.mark.gpu


# (d_in, d_out): one k-step, ragged columns over 1, 2 and 4 column parts and 4, 8
# and 16 waves, the longest normed row
@pytest.mark.parametrize("d_in,d_out", [(16, 1), (48, 33), (768, 250), (1024, 5224), (2064, 1000), (4096, 4097)])
@pytest.mark.parametrize("norm,accumulate", [(True, False), (True, True), (False, True), (False, False)])
def test_linear_row(d_in, d_out, norm, accumulate):
    import torch
    from mamba_hip.step import linear_row, pack_linear
    g = torch.Generator().manual_seed(d_in + d_out)
    w = torch.randn(d_in, d_out, generator=g).bfloat16()
    x = torch.randn(d_in, generator=g) * 3
    if not norm:
        x = x.bfloat16()
    gam, bias, y0 = (torch.randn(n, generator=g) for n in (d_in, d_out, d_out))
    out = y0.cuda() if accumulate else torch.empty(d_out, dtype=torch.bfloat16 if norm else torch.float32, device="cuda")
    linear_row(x.cuda(), pack_linear(w.cuda()), out, norm_w=gam.cuda() if norm else None, bias=bias.cuda(),
               accumulate=accumulate)
    torch.cuda.synchronize()
    n = x.double()
    if norm:
        n = n / (n.square().mean() + 8.1584695e-8).sqrt() * gam.double()
    want = n @ w.double() + bias.double() + (y0.double() if accumulate else 0)
    tol = (n.abs() @ w.double().abs()) * ((2.0 ** -9 if norm else 0) + 1e-5) + 1e-6 * (1 + want.abs())
    if out.dtype == torch.bfloat16:
        tol = tol + want.abs() * 2.0 ** -8
    assert bool(((out.cpu().double() - want).abs() <= tol).all())


@pytest.mark.parametrize("d_in", [48, 784, 1040])
def test_an_infinite_norm_weight_stays_in_its_products(d_in):
    """inf times a weight that is not zero is that infinity, not the NaN of a zero
    weight in the padding of some wave's last stage."""
    import torch
    from mamba_hip.step import linear_row, pack_linear
    d_out = 70
    g = torch.Generator().manual_seed(d_in)
    w = (torch.rand(d_in, d_out, generator=g) + 0.5).bfloat16() * (torch.randint(0, 2, (d_out,), generator=g) * 2 - 1)
    x = torch.rand(d_in, generator=g) + 0.5
    packed = pack_linear(w.cuda())
    for k in range(0, d_in, 16):
        gam = torch.ones(d_in)
        gam[k] = float("inf")
        out = torch.empty(d_out, device="cuda")
        linear_row(x.cuda(), packed, out, norm_w=gam.cuda())
        torch.cuda.synchronize()
        assert torch.equal(out.cpu(), w[k].float().sign() * float("inf")), k


def test_linear_row_refuses():
    import torch
    import mamba_hip
    from mamba_hip.step import linear_row, pack_linear
    dev = "cuda"
    w = pack_linear(torch.zeros(64, 64, device=dev))
    f, h, y = torch.zeros(64, device=dev), torch.zeros(64, device=dev, dtype=torch.bfloat16), torch.zeros(64, device=dev)
    long = torch.zeros(4112, device=dev)
    for args in ((f, None, y, False), (h, f, y, False), (torch.zeros(65, device=dev)[1:], f, y, False),
                 (h, None, h.clone(), True), (long, long, y, False)):
        with pytest.raises(mamba_hip.MambaHipError):
            linear_row(args[0], w, args[2], norm_w=args[1], accumulate=args[3])
