"""SSD calls on several streams at once, each with a workspace of its own."""

import pytest


def test_calls_share_no_workspace():
    from mamba_hip.ssd import workspace
    a, b = workspace("cpu", 1000), workspace("cpu", 1000)
    assert a.numel() >= 1000 and a.untyped_storage().data_ptr() != b.untyped_storage().data_ptr()


@pytest.mark.gpu
def test_two_streams():
    """Long sequences of few heads (segment states and packed fragments in the
    workspace) on two streams, then alone: the same bits."""
    import torch
    import mamba_hip
    b, l, h, p, n = 1, 3000, 8, 64, 128
    gen = torch.Generator(device="cuda").manual_seed(1)
    r = lambda *s: torch.randn(s, generator=gen, device="cuda")  # noqa: E731
    streams = [torch.cuda.Stream() for _ in range(2)]
    calls = []
    for io in (torch.bfloat16, torch.bfloat16, torch.float32, torch.float32):
        t = (r(b, l, h, p).to(io), torch.rand(b, l, h, generator=gen, device="cuda") * 0.1, -torch.ones(h, device="cuda"),
             r(b, l, 1, n).to(io) / 8, r(b, l, 1, n).to(io) / 8)
        dy = r(b, l, h, p).to(io)
        calls.append(lambda t=t: mamba_hip.ssd2_fwd(*t, chunk_len=256))
        calls.append(lambda t=t, dy=dy: tuple(v for v in mamba_hip.ssd2_bwd(dy, *t).values() if v is not None))
    want = [c() for c in calls]
    torch.cuda.synchronize()
    got = []
    for c in calls:
        pair = []
        for s in streams:
            with torch.cuda.stream(s):
                pair.append(c())
        got.append(pair)
    torch.cuda.synchronize()
    for w, pair in zip(want, got):
        for o in pair:
            assert all(torch.equal(x, y) for x, y in zip(w, o))
