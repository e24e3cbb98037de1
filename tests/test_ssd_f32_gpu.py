"""The segment-parallel f32-MFMA forward (ssd_f32.hip) of the Mamba-2 and
Mamba-3 seams at the edges of its chunks (64 fused rows), segments, headdim
blocks and ranks, vs the f64 oracle.

Tolerance: a result is a sum of at most a few hundred f32 products of O(1)
terms, each off by 2^-24 relative and by the 2^-22 of an exp of its decay, so
1e-5 of the row's scale bounds it; rtol 1e-4 is the f32 bar of the other tests.
bf16 results are rounded once, 2^-9."""

import numpy as np
import pytest

from inputs import bf16_round, ssd2_inputs, ssd3_inputs

pytestmark = pytest.mark.gpu

F32_TOL = dict(rtol=1e-4, atol=2e-5)
BF16_TOL = dict(rtol=2e-2, atol=1e-2)


def _dev(a, dtype=None):
    import torch
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).to("cuda", dtype)


# (b, l, h, p, g, n): one row, a chunk +- 1, several segments (few heads, long
# sequences), one segment (many heads), segments of two chunks, headdim blocks of
# 32 and of 64
CASES2 = [(1, 1, 2, 64, 1, 64), (1, 63, 4, 32, 2, 32), (2, 64, 2, 96, 1, 64), (1, 65, 2, 128, 2, 128),
          (1, 1500, 3, 64, 1, 128), (2, 640, 5, 192, 5, 32), (2, 130, 160, 64, 1, 64), (1, 4700, 3, 64, 1, 64)]


@pytest.mark.parametrize("dtype", ["f32", "bf16"])
@pytest.mark.parametrize("case", CASES2)
def test_ssd2(case, dtype):
    import torch
    import mamba_hip
    import oracle
    b, l, h, p, g, n = case
    inp = ssd2_inputs(seed=sum(case), b=b, l=l, h=h, p=p, g=g, n=n, h0=True)
    io = torch.float32
    if dtype == "bf16":
        io = torch.bfloat16
        for k in "xBC":
            inp[k] = bf16_round(inp[k])
    # x, B and C as column ranges of one row, as the block's conv output holds them
    rows = np.concatenate([inp["x"].reshape(b, l, -1), inp["B"].reshape(b, l, -1), inp["C"].reshape(b, l, -1)], 2)
    t = _dev(rows, io)
    x = t[:, :, :h * p].unflatten(2, (h, p))
    Bm = t[:, :, h * p:h * p + g * n].unflatten(2, (g, n))
    Cm = t[:, :, h * p + g * n:].unflatten(2, (g, n))
    y, hT = mamba_hip.ssd2_fwd(x, _dev(inp["dt"]), _dev(inp["A"]), Bm, Cm, _dev(inp["D"]), _dev(inp["h0"]), chunk_len=48)
    torch.cuda.synchronize()
    yr, hr = oracle.ssd2(inp["x"], inp["dt"], inp["A"], inp["B"], inp["C"], inp["D"], inp["h0"], chunk=64)
    tol = F32_TOL if dtype == "f32" else BF16_TOL
    np.testing.assert_allclose(y.float().cpu().numpy(), yr, **tol)
    np.testing.assert_allclose(hT.cpu().numpy(), hr, **F32_TOL)


# (b, l, m, h, p, n): ranks that fill a chunk with 64 / m steps, ragged ends,
# segments of two chunks
CASES3 = [(1, 33, 4, 2, 64, 64), (2, 15, 4, 2, 32, 128), (1, 300, 2, 3, 64, 128), (1, 3, 64, 2, 64, 64),
          (1, 257, 1, 4, 128, 32), (1, 70, 16, 2, 64, 128), (1, 710, 4, 12, 64, 128)]


@pytest.mark.parametrize("double", [False, True])
@pytest.mark.parametrize("case", CASES3)
def test_ssd3(case, double):
    import torch
    import mamba_hip
    import oracle
    b, l, m, h, p, n = case
    inp = ssd3_inputs(sum(case), b, l, m, h, p, n)
    v, da, B, C, h0 = (_dev(inp[k]) for k in ("v", "da", "B", "C", "h0"))
    if double:
        y, hT = mamba_hip.ssd3_double_fwd(v, da, B, C, h0, chunk_len=16)
        yr, hr = oracle.ssd3_double(inp["v"], inp["da"], inp["B"], inp["C"], inp["h0"], 16)
    else:
        y, hT = mamba_hip.ssd3_fwd(v, da, B, C, _dev(inp["gamma"]), _dev(inp["scale"]), h0, chunk_len=16)
        yr, hr = oracle.ssd3(inp["v"], inp["da"], inp["B"], inp["C"], inp["gamma"], inp["scale"], inp["h0"], 16)
    torch.cuda.synchronize()
    # sums over m ranks per step: the scale of y grows with sqrt(m)
    tol = dict(rtol=1e-4, atol=2e-5 * max(1.0, m ** 0.5))
    np.testing.assert_allclose(y.cpu().numpy(), yr, **tol)
    np.testing.assert_allclose(hT.cpu().numpy(), hr, **tol)


@pytest.mark.parametrize("l", [64, 200])
def test_ssd2_decays_after_a_reset(l):
    """A first half of 32 positions whose decays sum to 3200, then weak ones: the
    decay between two late positions is no difference of sums of that size
    (spacing 2^-12: 1e-4 off).  The late positions' own sums stay below 1, so that
    an exp is 2^-22 off and y a few times that: 1e-6 of its 2-norm, on whole and
    on split sequences."""
    import torch
    import mamba_hip
    import oracle
    b, h, p, n = 1, 2, 64, 64
    inp = ssd2_inputs(seed=l, b=b, l=l, h=h, p=p, g=1, n=n, h0=False)
    strong = np.arange(l) % 64 < 32
    inp["A"][:] = -1.0
    inp["dt"][:] = np.random.default_rng(l).uniform(0.01, 0.03, (b, l, h))
    inp["dt"][:, strong] = 100.0
    inp["x"][:, strong] *= np.float32(1e-4)  # dt weighs them
    t = {k: _dev(v) for k, v in inp.items()}
    y, hT = mamba_hip.ssd2_fwd(t["x"], t["dt"], t["A"], t["B"], t["C"], chunk_len=64)
    torch.cuda.synchronize()
    yr, hr = oracle.ssd2(inp["x"], inp["dt"], inp["A"], inp["B"], inp["C"], None, None, chunk=64)
    for got, ref in ((y.cpu().numpy()[:, ~strong], yr[:, ~strong]), (hT.cpu().numpy(), hr)):
        assert np.linalg.norm(got - ref) < 1e-6 * np.linalg.norm(ref)


@pytest.mark.parametrize("low", [np.finfo(np.float32).min, -np.inf])
@pytest.mark.parametrize("l,h", [(40, 2), (400, 2), (400, 160)])
def test_ssd3_decays_of_the_lowest_value(l, h, low):
    """Steps that forget everything before them, as masks set them, two of them in
    a chunk: their decay is 0 as exp(-1e4)'s is, and the rows after them have
    their own.  Whole and split sequences."""
    import torch
    import mamba_hip
    import oracle
    b, m, p, n = 1, 2, 64, 64
    inp = ssd3_inputs(l + h, b, l, m, h, p, n)
    reset = np.isin(np.arange(l) % 64, (5, 21))
    inp["da"][:, reset] = low
    t = {k: _dev(v) for k, v in inp.items()}
    y, hT = mamba_hip.ssd3_fwd(t["v"], t["da"], t["B"], t["C"], t["gamma"], t["scale"], t["h0"], chunk_len=64)
    torch.cuda.synchronize()
    inp["da"][:, reset] = -1e4
    yr, hr = oracle.ssd3(inp["v"], inp["da"], inp["B"], inp["C"], inp["gamma"], inp["scale"], inp["h0"], 16)
    np.testing.assert_allclose(y.cpu().numpy(), yr, rtol=1e-4, atol=3e-5)
    np.testing.assert_allclose(hT.cpu().numpy(), hr, rtol=1e-4, atol=3e-5)


def test_ssd3_infinite_value_of_the_last_step():
    """An infinite v gives infinities at its own row, as its product with C.B has
    it, and leaves the other columns alone."""
    import torch
    import mamba_hip
    b, l, m, h, p, n = 1, 3, 1, 1, 64, 64
    inp = ssd3_inputs(7, b, l, m, h, p, n)
    inp["v"][0, -1, 0, 0, 9] = np.inf
    t = {k: _dev(v) for k, v in inp.items()}
    y, _ = mamba_hip.ssd3_fwd(t["v"], t["da"], t["B"], t["C"], t["gamma"], t["scale"], t["h0"], chunk_len=16)
    torch.cuda.synchronize()
    y = y.cpu().numpy()[0, -1, 0, 0]
    cb = float(np.dot(inp["B"].reshape(l, n)[-1], inp["C"].reshape(l, n)[-1]))
    assert y[9] == np.sign(cb) * np.inf and np.isfinite(np.delete(y, 9)).all()


def test_ssd2_workspace_of_the_generic_path_still_serves():
    """A workspace of the SIMT kernels' size, without room for segment states,
    is accepted: the call then takes those kernels."""
    import ctypes

    import torch
    import mamba_hip
    from mamba_hip import _lib
    from mamba_hip.ssd import _ssd2_args, _stream
    b, l, h, p, n, q = 1, 700, 2, 64, 64, 512
    inp = ssd2_inputs(seed=3, b=b, l=l, h=h, p=p, g=1, n=n, h0=True)
    t = {k: _dev(v) for k, v in inp.items()}
    want = mamba_hip.ssd2_fwd(t["x"], t["dt"], t["A"], t["B"], t["C"], t["D"], t["h0"], chunk_len=q)
    nch = -(-l // q)
    small = torch.empty(-(-b * nch * h * p * n * 4 // 256) * 256 + 256, dtype=torch.uint8, device="cuda")
    y, hT = torch.empty_like(t["x"]), torch.empty_like(want[1])
    a = _ssd2_args(t["x"], t["dt"], t["A"], t["B"], t["C"], t["D"], t["h0"], None, q, y, hT)
    L = _lib.lib()
    assert L.mamba_ssd2_workspace_size(ctypes.byref(a)) > small.numel()
    _lib.check(L.mamba_ssd2_fwd(ctypes.byref(a), ctypes.c_void_p(small.data_ptr()), small.numel(), _stream("cuda")), "fwd")
    torch.cuda.synchronize()
    np.testing.assert_allclose(y.cpu().numpy(), want[0].cpu().numpy(), **F32_TOL)
    np.testing.assert_allclose(hT.cpu().numpy(), want[1].cpu().numpy(), **F32_TOL)
