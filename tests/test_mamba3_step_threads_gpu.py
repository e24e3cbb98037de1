"""mamba3_step_ssm with 512 threads per workgroup (small launches) against 256
(large ones): a row stepped alone against the row stepped inside a batch.  The
same sums in the same order, but the compiler contracts products into FMAs as it
likes in each form: a value made of at most 8 x 256 products may differ by that
many half-ulps of the largest, 2^11 2^-24 = 1.2e-4 of it."""

import pytest

pytestmark = pytest.mark.gpu


# the widest and the narrowest state rows, a headdim that leaves a ragged last
# pass in either form, ranks on both sides of the rule
@pytest.mark.parametrize("n,p,mimo,heads", [(128, 64, 4, 40), (256, 32, 8, 20), (8, 250, 1, 20), (64, 37, 2, 20),
                                            (16, 9, 4, 40), (32, 64, 1, 20)])
def test_rows_alone_equal_rows_in_a_batch(n, p, mimo, heads):
    import torch
    import mamba_hip
    b = 14  # 280 / 560 workgroups, past the rule's line; one row is far below it
    g = torch.Generator(device="cuda").manual_seed(n + p)
    cfg = mamba_hip.Mamba3Config(heads * p // 2, state_rank=n, mimo_rank=mimo,
                                 per_head_dim=p)
    m = cfg.init("cuda", torch.float32, g)
    H = cfg.nheads
    assert b * H > (512 if mimo == 4 else 256) >= H
    x = torch.randn(b, cfg.d_model, generator=g, device="cuda")
    cache = mamba_hip.Mamba3Cache(torch.randn(b, H, p, n, generator=g, device="cuda"),
                                  torch.randn(b, mimo, H, n, generator=g, device="cuda"),
                                  torch.randn(b, H, p, generator=g, device="cuda"),
                                  torch.randn(b, H, cfg.num_rope_angles, generator=g, device="cuda"))
    from mamba_hip.mamba3 import step_ssm, step_ssm_args
    proj = torch.randn(b, cfg.d_in_proj, generator=g, device="cuda")

    def run(rows):
        c = mamba_hip.Mamba3Cache(*(t[rows].clone() for t in (cache.ssm_bhpr, cache.k_state_bmhr, cache.v_state_bhp,
                                                              cache.angle_bha)))
        out = torch.empty(c.ssm_bhpr.shape[0], H * p, device="cuda")
        step_ssm(step_ssm_args(cfg, proj[rows].contiguous(), c, dt_bias=m.dt_bias, b_norm_w=m.b_norm_w,
                               c_norm_w=m.c_norm_w, b_bias=m.b_bias, c_bias=m.c_bias, D=m.D, mimo_x=m.mimo_x,
                               mimo_z=m.mimo_z, mimo_o=m.mimo_o, out_norm_w=m.out_norm_w, out=out), out.device, None)
        return out, c.ssm_bhpr, c.k_state_bmhr, c.v_state_bhp, c.angle_bha

    whole = run(slice(0, b))
    for i in (0, b - 1):
        for a, w in zip(run(slice(i, i + 1)), whole):
            assert float((a[0] - w[i]).abs().max()) <= 2.0 ** -13 * float(w.abs().max())
