"""The 8-wide mamba3_finish_fwd kernel (one dtype, headdim a multiple of 8)
at the edges of its split (1 and 8 positions per thread, ragged ends, ranks
kept in registers or not, out_norm over a head's lanes) vs the oracle.  The
oracle reads the bf16-rounded inputs; results are f32 sums of a few products
(rtol 1e-4, the f32 bar) or rounded once to bf16 (2^-9)."""

import numpy as np
import pytest

from inputs import bf16_round

pytestmark = pytest.mark.gpu


# (b, L, H, P, M, out_norm): the last two hold eight positions per thread
CASES = [(1, 1, 1, 8, 1, True), (2, 5, 3, 64, 2, True), (1, 7, 2, 40, 4, False), (1, 9, 2, 256, 8, True),
         (3, 6, 5, 128, 1, False), (1, 16387, 32, 64, 1, False), (2, 8195, 16, 128, 4, True)]


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("case", CASES)
def test_finish(case, dtype):
    import torch
    import mamba_hip
    import oracle
    b, L, H, P, M, norm = case
    rng = np.random.default_rng(sum(case))
    f = lambda *s: rng.standard_normal(s, dtype=np.float32)  # noqa: E731
    rnd, io = (bf16_round, torch.bfloat16) if dtype == "bf16" else (lambda a: a, torch.float32)
    y, v, zw = rnd(f(b, L, M, H, P)), rnd(f(b, L, M, H, P)), rnd(f(b, L, H * P + 16))
    D, mz, mo, onw = f(H), f(H, M, P), f(H, M, P), f(P)
    g = lambda a, t=torch.float32: torch.from_numpy(np.ascontiguousarray(a)).cuda().to(t)  # noqa: E731
    cfg = mamba_hip.Mamba3Config(d_model=H * P // 2 or 1, per_head_dim=P, mimo_rank=M)
    out = mamba_hip.mamba3_finish_fwd(cfg, g(y, io), g(v, io), g(zw, io)[:, :, :H * P], D=g(D),
                                      mimo_z=g(mz) if M > 1 else None, mimo_o=g(mo) if M > 1 else None,
                                      out_norm_w=g(onw) if norm else None)
    torch.cuda.synchronize()
    want = oracle.mamba3_finish_fwd(y, v, zw[:, :, :H * P], dict(D=D, mimo_z=mz, mimo_o=mo,
                                                                 out_norm_w=onw if norm else None))
    tol = dict(rtol=1e-4, atol=2e-5) if dtype == "f32" else dict(rtol=1e-2, atol=1e-2)
    np.testing.assert_allclose(out.float().cpu().numpy(), want, **tol)


def test_gate_divides_as_the_general_kernel_does():
    """bf16, one rank, no norm: both kernels form y z / (1 + exp(-z)) in f32 and
    round once, so that they agree bit for bit (a reciprocal 1 ulp off would turn
    about one bf16 rounding in 2^17: some 60 of these 8 million)."""
    import torch
    import mamba_hip
    b, L, H, P = 2, 8192, 8, 64
    gen = torch.Generator(device="cuda").manual_seed(3)
    y = torch.randn(b, L, 1, H, P, device="cuda", generator=gen).bfloat16()
    z = (4 * torch.randn(b, L, H * P, device="cuda", generator=gen)).bfloat16()
    cfg = mamba_hip.Mamba3Config(d_model=H * P // 2, per_head_dim=P, mimo_rank=1)
    out = mamba_hip.mamba3_finish_fwd(cfg, y, None, z)
    odd = torch.empty(b * L * H * P + 1, device="cuda", dtype=torch.bfloat16)[1:].view(b, L, H * P)
    mamba_hip.mamba3_finish_fwd(cfg, y, None, z, out=odd)  # rows off 16 bytes: the general kernel
    torch.cuda.synchronize()
    assert torch.equal(out, odd)
