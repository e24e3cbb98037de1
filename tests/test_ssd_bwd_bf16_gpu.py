"""The SSD backwards on bf16 rows read in place against the same rows widened to
f32 first: the same arithmetic on the same values, so they differ by the
compiler's choice of FMAs alone (sums of up to 2^9 products: 2^9 2^-24 = 3e-5 of
the largest)."""

import pytest

pytestmark = pytest.mark.gpu


def _same(a, b):
    for k, w in b.items():
        assert (w is None) == (a[k] is None)
        if w is not None:
            assert a[k].dtype == w.dtype and float((a[k] - w).abs().max()) <= 3e-5 * float(w.abs().max()) + 1e-30, k


# one step, a ragged chunk, several segments, one that ends in half a chunk; both dstates; grouped; rows that only
# the f32 route takes (odd offset, every other value, headdim 32)
@pytest.mark.parametrize("l,h,g,p,n,form", [(1, 4, 1, 64, 64, "plain"), (65, 4, 2, 64, 128, "plain"), (700, 2, 1, 64, 128, "plain"), (70, 200, 1, 64, 128, "plain"),
                                            (300, 2, 2, 64, 64, "wide"), (70, 4, 1, 64, 64, "odd"),
                                            (70, 4, 1, 64, 128, "every other"), (70, 4, 1, 32, 64, "plain")])
def test_mamba2(l, h, g, p, n, form):
    import torch
    import mamba_hip
    r = torch.Generator(device="cuda").manual_seed(l + n)

    def rows(*s):
        if form == "wide":
            return torch.randn(*s[:-1], s[-1] + 4, generator=r, device="cuda").bfloat16()[..., :s[-1]]
        if form == "odd":
            return torch.randn(*s[:-1], s[-1] + 4, generator=r, device="cuda").bfloat16()[..., 1:s[-1] + 1]
        if form == "every other":
            return torch.randn(*s[:-1], 2 * s[-1], generator=r, device="cuda").bfloat16()[..., ::2]
        return torch.randn(*s, generator=r, device="cuda").bfloat16()

    x, dy, B, C = rows(2, l, h, p), rows(2, l, h, p), rows(2, l, g, n), rows(2, l, g, n)
    dt = torch.rand(2, l, h, generator=r, device="cuda") * 0.1
    A, D = -torch.rand(h, generator=r, device="cuda") * 8, torch.randn(h, generator=r, device="cuda")
    h0, dh = (torch.randn(2, h, p, n, generator=r, device="cuda") for _ in range(2))
    _same(mamba_hip.ssd2_bwd(dy, x, dt, A, B, C, D, h0, dh),
          mamba_hip.ssd2_bwd(dy.float(), x.float(), dt, A, B.float(), C.float(), D, h0, dh))


@pytest.mark.parametrize("l,m,h,n,weights", [(1, 4, 2, 64, True), (33, 4, 2, 128, True), (300, 1, 2, 128, False),
                                             (40, 8, 2, 64, True)])
def test_mamba3(l, m, h, n, weights):
    import torch
    import mamba_hip
    r = torch.Generator(device="cuda").manual_seed(l + n)
    v, dy = (torch.randn(2, l, m, h, 64, generator=r, device="cuda").bfloat16() for _ in range(2))
    B, C = (torch.randn(2, l, m, h, n, generator=r, device="cuda").bfloat16() for _ in range(2))
    da = -torch.rand(2, l, h, generator=r, device="cuda")
    ga, sc = (torch.rand(2, l, h, generator=r, device="cuda") if weights else None for _ in range(2))
    h0, dh = (torch.randn(2, h, 64, n, generator=r, device="cuda") for _ in range(2))
    _same(mamba_hip.ssd3_bwd(dy, v, da, B, C, ga, sc, h0, dh),
          mamba_hip.ssd3_bwd(dy.float(), v.float(), da, B.float(), C.float(), ga, sc, h0, dh))
