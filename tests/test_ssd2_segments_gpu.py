"""The bf16 SSD forward split into sequence segments (ssd2_seg_state, then the
scan of every segment) vs the oracle: few heads and long or ragged sequences,
both state widths and chunk lengths, segments of one chunk and of several with
each head set, decays that underflow from chunk to chunk, initial states, and a
workspace without room for segments (one segment).  bf16 bars of the other
forward tests; states accumulate bf16 products in f32."""

import numpy as np
import pytest

from inputs import bf16_round, ssd2_inputs

pytestmark = pytest.mark.gpu

TOL = dict(rtol=2e-2, atol=1e-2)


def _dev(inp):
    import torch
    io = torch.bfloat16
    return {k: None if v is None else torch.from_numpy(v).cuda().to(io if k in "xBC" else torch.float32)
            for k, v in inp.items()}


# (b, l, h, g, n, chunk, dt range): two chunks and a full chip, which stay whole,
# and segments of one chunk (of three in the fourth), ragged ends, chunks of 32
CASES = [(1, 65, 1, 1, 128, 64, (1e-3, 0.1)), (1, 1000, 2, 1, 64, 64, (1e-3, 0.1)), (2, 777, 4, 1, 128, 256, (1e-3, 0.1)),
         (1, 2049, 10, 2, 128, 256, (1e-3, 0.1)), (1, 500, 3, 3, 64, 32, (1e-3, 0.1)),
         (1, 640, 4, 1, 128, 64, (2.0, 8.0)), (3, 300, 80, 1, 128, 256, (1e-3, 0.1))]


# (b, l, h, g, n, chunk): segments of 2 or 3 chunks, the last one shorter or with
# a ragged chunk, at head sets of 1 (with chunks of 64 and of 32), 2, 4 and 5
SPLIT = [(1, 2950, 1, 1, 64, 64), (1, 1500, 3, 3, 64, 32), (1, 4500, 6, 1, 128, 64), (1, 2600, 8, 1, 128, 256),
         (2, 2049, 20, 2, 128, 256)]


# decay 40: A of -40 to -640, so that most steps underflow over a chunk and many by
# themselves.  dt stays small: y holds dt (C.B) x, whose operands' roundings, 2^-8
# together, pass atol at a dt of 8 (|C.B| <= 0.4, |x| <= 4.5: 0.05).
@pytest.mark.parametrize("case", SPLIT)
@pytest.mark.parametrize("decay", [1, 40])
def test_segments_of_several_chunks_match_oracle(case, decay):
    _check(*case, (1e-3, 0.1), decay)


@pytest.mark.parametrize("case", SPLIT)
def test_these_sequences_split(case):
    """A workspace for the packed fragments alone keeps a sequence whole, which
    rounds its final state elsewhere than segments do."""
    import torch
    import mamba_hip
    b, l, h, g, n, q = case
    t = _dev(ssd2_inputs(seed=1, b=b, l=l, h=h, p=64, g=g, n=n, h0=True))
    _, hT = mamba_hip.ssd2_fwd(t["x"], t["dt"], t["A"], t["B"], t["C"], t["D"], t["h0"], chunk_len=q)
    rows = min(q, 64)
    T, nk, ks = rows // 32, n // 16, rows // 16
    _, whole = _with_workspace(t, q, b * -(-l // rows) * g * (T * (T + 1) + T * nk + n // 32 * ks) * 1024)
    torch.cuda.synchronize()
    assert not torch.equal(hT, whole)
    torch.testing.assert_close(hT, whole, **TOL)


def _with_workspace(t, q, nbytes):
    import ctypes

    import torch
    from mamba_hip import _lib
    from mamba_hip.ssd import _ssd2_args, _stream
    y, hT = torch.empty_like(t["x"]), torch.empty_like(t["h0"])
    a = _ssd2_args(t["x"], t["dt"], t["A"], t["B"], t["C"], t["D"], t["h0"], None, q, y, hT)
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    _lib.check(_lib.lib().mamba_ssd2_fwd(ctypes.byref(a), ctypes.c_void_p(ws.data_ptr()), nbytes, _stream("cuda")), "fwd")
    return y, hT


@pytest.mark.parametrize("case", CASES)
def test_segments_match_oracle(case):
    _check(*case)


def _check(b, l, h, g, n, q, dtr, decay=1):
    import torch
    import mamba_hip
    import oracle
    inp = ssd2_inputs(seed=l, b=b, l=l, h=h, p=64, g=g, n=n, h0=True, dt_range=dtr)
    inp["A"] *= np.float32(decay)
    for k in "xBC":
        inp[k] = bf16_round(inp[k])
    t = _dev(inp)
    hpr = torch.full((h, 64, n), 0.05, device="cuda")
    y, hT = mamba_hip.ssd2_fwd(t["x"], t["dt"], t["A"], t["B"], t["C"], t["D"], t["h0"], hpr, chunk_len=q)
    torch.cuda.synchronize()
    yr, hr = oracle.ssd2(inp["x"], inp["dt"], inp["A"], inp["B"], inp["C"], inp["D"], inp["h0"] + np.float32(0.05), chunk=64)
    np.testing.assert_allclose(y.float().cpu().numpy(), yr, **TOL)
    np.testing.assert_allclose(hT.cpu().numpy(), hr, **TOL)


def test_workspace_without_segments():
    import ctypes

    import torch
    import mamba_hip
    from mamba_hip import _lib
    from mamba_hip.ssd import _ssd2_args, _stream
    b, l, h, n, q = 1, 900, 4, 128, 256
    t = _dev(ssd2_inputs(seed=1, b=b, l=l, h=h, p=64, g=1, n=n, h0=True))
    want = mamba_hip.ssd2_fwd(t["x"], t["dt"], t["A"], t["B"], t["C"], t["D"], t["h0"], chunk_len=q)
    y, hT = torch.empty_like(t["x"]), torch.empty_like(want[1])
    a = _ssd2_args(t["x"], t["dt"], t["A"], t["B"], t["C"], t["D"], t["h0"], None, q, y, hT)
    L = _lib.lib()
    # 38 KB of packed fragments per chunk of 64 positions: C.B^T 6, C 16, B 16
    least = -(-l // 64) * 38 * 1024
    assert L.mamba_ssd2_workspace_size(ctypes.byref(a)) > least
    ws = torch.empty(least, dtype=torch.uint8, device="cuda")
    _lib.check(L.mamba_ssd2_fwd(ctypes.byref(a), ctypes.c_void_p(ws.data_ptr()), least, _stream("cuda")), "fwd")
    torch.cuda.synchronize()
    np.testing.assert_allclose(y.float().cpu().numpy(), want[0].float().cpu().numpy(), **TOL)
    np.testing.assert_allclose(hT.cpu().numpy(), want[1].cpu().numpy(), rtol=1e-2, atol=1e-3)
