"""final_state may be the memory of initial_state: a cache updated in place.  Where a
sequence is split into segments that run side by side, the last one writes while
others still start; the result is bit for bit that of separate tensors.  Each
case is sized to split, which its workspace or its rounding shows."""

import ctypes

import numpy as np
import pytest

from inputs import ssd2_inputs, ssd3_inputs

pytestmark = pytest.mark.gpu


def _dev(a, dtype=None):
    import torch
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dtype)


def _in_place(run, h0):
    """run(initial_state, final_state) -> (y, final_state)"""
    import torch
    y, hT = run(h0, torch.empty_like(h0))
    torch.cuda.synchronize()
    y, hT = y.clone(), hT.clone()
    cache = h0.clone()
    y2, hT2 = run(cache, cache)
    torch.cuda.synchronize()
    assert hT2.data_ptr() == cache.data_ptr()
    assert torch.equal(y, y2) and torch.equal(hT, hT2)


# (b, l, h, p, n): many segments of a chunk each, and of several chunks (headdim
# blocks of 32)
@pytest.mark.parametrize("case", [(1, 1500, 2, 64, 64), (1, 6000, 3, 96, 128)])
def test_ssd2_f32(case):
    import mamba_hip
    from mamba_hip import _lib
    from mamba_hip.ssd import _ssd2_args
    b, l, h, p, n = case
    q = 512
    t = {k: _dev(v) for k, v in ssd2_inputs(seed=l, b=b, l=l, h=h, p=p, g=1, n=n, h0=True).items()}
    a = _ssd2_args(t["x"], t["dt"], t["A"], t["B"], t["C"], t["D"], t["h0"], None, q, t["x"], t["h0"])
    simt = -(-l // q) * (b * h * p * n + h) * 4 + 512  # the SIMT kernels' workspace at most
    assert _lib.lib().mamba_ssd2_workspace_size(ctypes.byref(a)) > simt
    _in_place(lambda h0, hT: mamba_hip.ssd2_fwd(t["x"], t["dt"], t["A"], t["B"], t["C"], t["D"], h0, chunk_len=q,
                                                final_state=hT), t["h0"])


@pytest.mark.parametrize("double", [False, True])
def test_ssd3_f32(double):
    import mamba_hip
    from mamba_hip import _lib
    from mamba_hip.ssd3 import _args
    l, q = 700, 64
    t = {k: _dev(v) for k, v in ssd3_inputs(5, 1, l, 4, 2, 64, 128).items()}
    v, da, B, C = (t[k] for k in ("v", "da", "B", "C"))
    a = _args(v, da, B, C, t["gamma"], t["scale"], t["h0"], q, v, t["h0"])
    simt = -(-l // q) * (2 * 64 * 128 + 2) * 4 + 512  # the SIMT kernels' workspace at most
    assert _lib.lib().mamba_ssd3_workspace_size(ctypes.byref(a)) > simt
    if double:
        _in_place(lambda h0, hT: mamba_hip.ssd3_double_fwd(v, da, B, C, h0, q, final_state=hT), t["h0"])
    else:
        _in_place(lambda h0, hT: mamba_hip.ssd3_fwd(v, da, B, C, t["gamma"], t["scale"], h0, q, final_state=hT), t["h0"])


# (b, l, h, n, chunk): segments of one chunk of 64 positions, of several, of
# chunks of 32
@pytest.mark.parametrize("case", [(1, 1000, 2, 64, 64), (1, 5000, 8, 128, 256), (2, 700, 4, 128, 32)])
@pytest.mark.parametrize("hpr", [False, True])
def test_ssd2_bf16(case, hpr):
    import torch
    import mamba_hip
    from mamba_hip import _lib
    from mamba_hip.ssd import _ssd2_args, _stream
    b, l, h, n, q = case
    t = {k: _dev(v, torch.bfloat16 if k in "xBC" else None)
         for k, v in ssd2_inputs(seed=l, b=b, l=l, h=h, p=64, g=1, n=n, h0=True).items()}
    add = torch.full((h, 64, n), 0.05, device="cuda") if hpr else None
    # a workspace with room for the packed operand fragments (1 KB each) alone: the
    # sequence whole, rounded elsewhere than in segments
    rows = 32 if q == 32 else 64
    T, nk, ks = rows // 32, n // 16, rows // 16
    least = b * -(-l // rows) * (T * (T + 1) + T * nk + n // 32 * ks) * 1024
    y, hT = torch.empty_like(t["x"]), torch.empty_like(t["h0"])
    a = _ssd2_args(t["x"], t["dt"], t["A"], t["B"], t["C"], t["D"], t["h0"], add, q, y, hT)
    ws = torch.empty(least, dtype=torch.uint8, device="cuda")
    _lib.check(_lib.lib().mamba_ssd2_fwd(ctypes.byref(a), ctypes.c_void_p(ws.data_ptr()), least, _stream("cuda")), "fwd")
    split = mamba_hip.ssd2_fwd(t["x"], t["dt"], t["A"], t["B"], t["C"], t["D"], t["h0"], add, chunk_len=q)
    torch.cuda.synchronize()
    assert not torch.equal(hT, split[1])
    _in_place(lambda h0, hT: mamba_hip.ssd2_fwd(t["x"], t["dt"], t["A"], t["B"], t["C"], t["D"], h0, add, chunk_len=q,
                                                final_state=hT), t["h0"])
