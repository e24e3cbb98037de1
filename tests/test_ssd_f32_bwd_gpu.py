"""The segment-parallel f32-MFMA backward (ssd_f32_bwd.hip) of the Mamba-2 and
Mamba-3 seams at the edges of its chunks (64 fused rows), segments, ranks and
the two state widths, vs the float64 reverse recurrence (oracle.ssd2_bwd,
oracle.ssd3_bwd): f32 gradients within rtol 1e-4 and an absolute 1e-4 of each
gradient's scale, the bars of the other backward tests."""

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _t(a):
    import torch
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _close(got, want, name):
    scale = float(np.abs(want).max()) or 1.0
    np.testing.assert_allclose(got.cpu().numpy(), want, rtol=1e-4, atol=1e-4 * scale, err_msg=name)


# (b, l, h, g, n, optional): one row, half a chunk (also as the last one of a whole
# sequence) and a chunk +- 1, many segments (one head),
# segments of two chunks, per-head and grouped B / C, with and without D, h0 and
# d(final state)
CASES2 = [(1, 1, 2, 1, 64, True), (2, 63, 2, 2, 64, False), (1, 64, 3, 1, 128, True), (1, 65, 2, 1, 64, True),
          (1, 700, 1, 1, 128, True), (2, 333, 4, 2, 64, True), (1, 130, 300, 1, 64, False), (1, 2500, 12, 2, 64, True),
          (2, 31, 2, 2, 64, True), (1, 32, 4, 2, 128, True), (2, 33, 2, 1, 128, True), (1, 90, 200, 2, 128, True)]


@pytest.mark.parametrize("case", CASES2)
def test_ssd2(case):
    import torch
    import mamba_hip
    b, l, h, g, n, opt = case
    p = 64
    rng = np.random.default_rng(sum(case))
    r = lambda *s: rng.standard_normal(s, dtype=np.float32)  # noqa: E731
    x, dy, B, C = r(b, l, h, p), r(b, l, h, p), r(b, l, g, n) / np.float32(n ** 0.5), r(b, l, g, n) / np.float32(n ** 0.5)
    dt = rng.uniform(0.01, 0.3, (b, l, h)).astype(np.float32)
    A = (-np.exp(rng.uniform(0.0, np.log(8.0), h))).astype(np.float32)
    D, h0, dF = (r(h), 0.3 * r(b, h, p, n), r(b, h, p, n)) if opt else (None, None, None)
    out = mamba_hip.ssd2_bwd(_t(dy), _t(x), _t(dt), _t(A), _t(B), _t(C), _t(D), _t(h0), _t(dF))
    torch.cuda.synchronize()
    want = oracle.ssd2_bwd(dy, dF, x, dt, A, B, C, D, h0)
    for k, w in (("dx", "dx"), ("ddt", "ddt"), ("dA", "dA"), ("dB", "dB"), ("dC", "dC"), ("d_initial_state", "dh0")):
        _close(out[k], want[w], k)
    if opt:
        _close(out["dD"], want["dD"], "dD")


# (b, l, m, h, g, n, optional): 64 / m steps per chunk, ragged ends, segments of
# two chunks, the double seam's unit weights (optional False)
CASES3 = [(1, 33, 4, 2, 2, 64, True), (1, 3, 32, 2, 1, 64, True), (2, 100, 2, 2, 1, 128, True),
          (1, 400, 4, 1, 1, 64, True), (1, 129, 1, 3, 3, 64, False), (1, 17, 16, 2, 2, 128, False), (1, 710, 4, 12, 1, 64, True),
          (2, 8, 4, 2, 1, 128, True), (1, 9, 4, 2, 1, 128, True), (2, 1, 32, 2, 1, 64, True), (1, 24, 4, 200, 1, 128, True)]


@pytest.mark.parametrize("case", CASES3)
def test_ssd3(case):
    import torch
    import mamba_hip
    b, l, m, h, g, n, opt = case
    p = 64
    rng = np.random.default_rng(sum(case))
    r = lambda *s: rng.standard_normal(s, dtype=np.float32)  # noqa: E731
    v, dy = r(b, l, m, h, p), r(b, l, m, h, p)
    B, C = r(b, l, m, g, n) / np.float32(n ** 0.5), r(b, l, m, g, n) / np.float32(n ** 0.5)
    da = -rng.uniform(0.01, 0.5, (b, l, h)).astype(np.float32)
    gam, scl = (rng.uniform(0.01, 0.3, (b, l, h)).astype(np.float32) for _ in range(2)) if opt else (None, None)
    h0, dF = (0.3 * r(b, h, p, n), r(b, h, p, n)) if opt else (None, None)
    out = mamba_hip.ssd3_bwd(_t(dy), _t(v), _t(da), _t(B), _t(C), _t(gam), _t(scl), _t(h0), _t(dF))
    torch.cuda.synchronize()
    want = oracle.ssd3_bwd(dy, dF, v, da, B, C, gam, scl, h0)
    for k, w in (("dv", "dv"), ("dda", "dda"), ("dB", "dB"), ("dC", "dC"), ("d_initial_state", "dh0")):
        _close(out[k], want[w], k)
    if opt:
        _close(out["dgamma"], want["dgamma"], "dgamma")
        _close(out["dscale"], want["dscale"], "dscale")


@pytest.mark.parametrize("l,h", [(64, 2), (200, 2), (200, 300)])
def test_ssd2_decays_after_a_reset(l, h):
    """A first half of 32 positions whose decays sum to 3200, then weak ones: the
    decay between two late positions is no difference of sums of that size
    (spacing 2^-12: 1e-4 off).  The late rows' own sums stay below 1, so that an
    exp is 2^-23 off and a gradient a few times that: 2e-6 of its 2-norm, on
    whole and on split sequences."""
    import torch
    import mamba_hip
    b, g, n, p = 1, 1, 64, 64
    rng = np.random.default_rng(l)
    r = lambda *s: rng.standard_normal(s, dtype=np.float32)  # noqa: E731
    x, dy, B, C = r(b, l, h, p), r(b, l, h, p), r(b, l, g, n) / 8, r(b, l, g, n) / 8
    dt = rng.uniform(0.01, 0.03, (b, l, h)).astype(np.float32)
    dt[:, np.arange(l) % 64 < 32] = 100.0
    A = np.full(h, -1.0, np.float32)
    x[:, np.arange(l) % 64 < 32] *= 1e-4  # dt weighs them
    out = mamba_hip.ssd2_bwd(_t(dy), _t(x), _t(dt), _t(A), _t(B), _t(C))
    torch.cuda.synchronize()
    want = oracle.ssd2_bwd(dy, None, x, dt, A, B, C, None, None)
    late = np.arange(l) % 64 >= 32
    for k in ("dx", "dB", "dC"):
        got, ref = out[k].cpu().numpy()[:, late].astype(np.float64), want[k][:, late]
        err = np.linalg.norm(got - ref) / np.linalg.norm(ref)
        assert err < 2e-6, (k, err)


@pytest.mark.parametrize("low", [np.finfo(np.float32).min, -np.inf])
@pytest.mark.parametrize("l", [40, 400])
def test_ssd3_decays_of_the_lowest_value(l, low):
    """Steps that forget everything before them, as masks set them, two of them in
    a chunk: the gradients are those of a decay of exp(-1e4), which is 0."""
    import torch
    import mamba_hip
    b, m, h, g, n, p = 1, 2, 2, 1, 64, 64
    rng = np.random.default_rng(l)
    r = lambda *s: rng.standard_normal(s, dtype=np.float32)  # noqa: E731
    v, dy, B, C = r(b, l, m, h, p), r(b, l, m, h, p), r(b, l, m, g, n) / 8, r(b, l, m, g, n) / 8
    da = -rng.uniform(0.01, 0.5, (b, l, h)).astype(np.float32)
    gam, scl = (rng.uniform(0.01, 0.3, (b, l, h)).astype(np.float32) for _ in range(2))
    h0, dF = 0.3 * r(b, h, p, n), r(b, h, p, n)
    reset = np.isin(np.arange(l) % 64, (5, 21))
    da[:, reset] = low
    out = mamba_hip.ssd3_bwd(_t(dy), _t(v), _t(da), _t(B), _t(C), _t(gam), _t(scl), _t(h0), _t(dF))
    torch.cuda.synchronize()
    da[:, reset] = -1e4
    want = oracle.ssd3_bwd(dy, dF, v, da, B, C, gam, scl, h0)
    for k, w in (("dv", "dv"), ("dda", "dda"), ("dB", "dB"), ("dC", "dC"), ("d_initial_state", "dh0"),
                 ("dgamma", "dgamma"), ("dscale", "dscale")):
        _close(out[k], want[w], k)


def test_ssd3_infinite_dy_of_the_first_step():
    """An infinite dy gives infinities in its own step's dv, as its product with
    C.B has it, and leaves the other columns of dv alone."""
    import torch
    import mamba_hip
    b, l, m, h, g, n, p = 1, 1, 1, 1, 1, 64, 64
    rng = np.random.default_rng(1)
    r = lambda *s: rng.standard_normal(s, dtype=np.float32)  # noqa: E731
    v, dy, B, C = r(b, l, m, h, p), r(b, l, m, h, p), r(b, l, m, g, n), r(b, l, m, g, n)
    dy[..., 9] = np.inf
    da, gam, scl = (-np.ones((b, l, h), np.float32), np.ones((b, l, h), np.float32), np.ones((b, l, h), np.float32))
    out = mamba_hip.ssd3_bwd(_t(dy), _t(v), _t(da), _t(B), _t(C), _t(gam), _t(scl))
    torch.cuda.synchronize()
    dv = out["dv"].cpu().numpy().reshape(p)
    assert dv[9] == np.sign(float((B * C).sum())) * np.inf and np.isfinite(np.delete(dv, 9)).all()


def test_ssd2_any_segment_count_gives_the_same_gradients():
    """A workspace that holds fewer segments (as small as the SIMT kernels', one
    entry state per 32 positions) is used with fewer; both agree to f32 rounding."""
    import ctypes

    import torch
    import mamba_hip
    from mamba_hip import _lib
    b, l, h, n, p = 1, 1000, 2, 64, 64
    rng = np.random.default_rng(11)
    r = lambda *s: rng.standard_normal(s, dtype=np.float32)  # noqa: E731
    t = {k: _t(v) for k, v in dict(dy=r(b, l, h, p), x=r(b, l, h, p), dt=rng.uniform(0.01, 0.3, (b, l, h)).astype(np.float32),
                                   A=-np.ones(h, np.float32), B=r(b, l, h, n) / 8, C=r(b, l, h, n) / 8).items()}
    ref = mamba_hip.ssd2_bwd(t["dy"], t["x"], t["dt"], t["A"], t["B"], t["C"])
    a = _lib.Ssd2BwdArgs()
    a.batch, a.seqlen, a.nheads, a.headdim, a.ngroups, a.dstate = b, l, h, p, h, n
    out = {k: torch.empty_like(ref[k]) for k in ("dx", "ddt", "dA", "dB", "dC", "d_initial_state")}
    for k, v in list(t.items()) + list(out.items()):
        setattr(a, k, v.data_ptr())
    for k, w in (("x", p), ("dy", p), ("B", n), ("C", n)):
        q = "g" if k in "BC" else "h"
        for nm, s in ((f"{k}_sb", l * h * w), (f"{k}_sl", h * w), (f"{k}_s{q}", w)):
            setattr(a, nm, s)
    a.dt_sb, a.dt_sl, a.dt_sh = l * h, h, 1
    L = _lib.lib()
    full = L.mamba_ssd2_bwd_workspace_size(ctypes.byref(a))
    ws = torch.empty(full, dtype=torch.uint8, device="cuda")
    state = h * p * n * 4
    assert full > 32 * state + 512
    for nbytes in (32 * state + 512, full):
        _lib.check(L.mamba_ssd2_bwd(ctypes.byref(a), ctypes.c_void_p(ws.data_ptr()), nbytes,
                                    ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "bwd")
        torch.cuda.synchronize()
        for k in out:
            _close(out[k], ref[k].cpu().numpy(), f"{k} in {nbytes} bytes")
