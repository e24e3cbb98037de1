"""final_state may be the memory of initial_state (a cache updated in place), and
d_initial_state that of d_final_state.  Where a sequence is split into segments
that run side by side, one writes while others still start; the result is bit for bit that of separate tensors.  Each
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


# (b, l, h, n): segments of one chunk and of several
@pytest.mark.parametrize("case", [(1, 1000, 2, 64), (2, 2500, 6, 128)])
def test_ssd2_bwd(case):
    import torch
    from mamba_hip import _lib
    from mamba_hip.ssd import _stream
    b, l, h, n = case
    p = 64
    rng = np.random.default_rng(l)
    r = lambda *s: _dev(rng.standard_normal(s, dtype=np.float32))  # noqa: E731
    t = dict(dy=r(b, l, h, p), x=r(b, l, h, p), dt=_dev(rng.uniform(0.01, 0.3, (b, l, h)).astype(np.float32)),
             A=-torch.ones(h, device="cuda"), B=r(b, l, 1, n) / 8, C=r(b, l, 1, n) / 8, initial_state=r(b, h, p, n))
    dF = r(b, h, p, n)
    a = _lib.Ssd2BwdArgs()
    a.batch, a.seqlen, a.nheads, a.headdim, a.ngroups, a.dstate = b, l, h, p, 1, n
    for k in ("x", "dy"):
        for nm, v in (("sb", l * h * p), ("sl", h * p), ("sh", p)):
            setattr(a, f"{k}_{nm}", v)
    for k in ("B", "C"):
        for nm, v in (("sb", l * n), ("sl", n), ("sg", n)):
            setattr(a, f"{k}_{nm}", v)
    a.dt_sb, a.dt_sl, a.dt_sh = l * h, h, 1
    for k, v in t.items():
        setattr(a, k, v.data_ptr())
    L = _lib.lib()

    def run(d_final, d_initial, nbytes):
        out = {k: torch.empty_like(t[s]) for k, s in (("dx", "x"), ("ddt", "dt"), ("dA", "A"), ("dB", "B"), ("dC", "C"))}
        for k, v in out.items():
            setattr(a, k, v.data_ptr())
        a.d_final_state, a.d_initial_state = d_final.data_ptr(), d_initial.data_ptr()
        _lib.check(L.mamba_ssd2_bwd(ctypes.byref(a), ctypes.c_void_p(ws.data_ptr()), nbytes, _stream("cuda")), "bwd")
        torch.cuda.synchronize()
        return dict(out, dh0=d_initial)

    for k in ("dx", "ddt", "dA", "dB", "dC", "d_initial_state"):  # the size query wants every pointer
        setattr(a, k, dF.data_ptr())
    full = L.mamba_ssd2_bwd_workspace_size(ctypes.byref(a))
    ws = torch.empty(full, dtype=torch.uint8, device="cuda")
    want = run(dF, torch.empty_like(dF), full)
    cache = dF.clone()
    got = run(cache, cache, full)
    for k in want:
        assert torch.equal(got[k], want[k]), k
    # the SIMT kernels' size (a state per 32 positions, dB and dC per head, partial
    # sums) holds fewer segments: rounded elsewhere, so that full does split
    nch = -(-l // 32)
    fewer = (b * h * nch * p * n + 2 * b * l * h * n) * 4 + 4 * 256 + 2 * b * h * 4
    assert fewer < full
    assert not torch.equal(run(dF, torch.empty_like(dF), fewer)["dx"], want["dx"])
