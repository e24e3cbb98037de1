"""mamba1_scan in time segments and over rows at odd addresses, vs the float64
oracle at the other scan tests' tolerance (f32 sums of terms that
a decay below 1 weighs)."""

import numpy as np
import pytest

from inputs import mamba1_inputs

pytestmark = pytest.mark.gpu
TOL = dict(rtol=1e-4, atol=2e-5)


# one tile (no split), a last tile of one token, whole tiles, many segments whose
# last is short, 16-byte rows and odd ones; ws: segments the workspace holds
@pytest.mark.parametrize("gate", [True, False])
@pytest.mark.parametrize("l,ws", [(31, None), (33, None), (96, None), (97, 2), (515, None), (512, 5), (515, 1), (515, 0)])
def test_segments_match_oracle(l, ws, gate, monkeypatch):
    import torch
    import mamba_hip
    import oracle
    from mamba_hip import _lib
    b, d, n = 2, 70, 16
    inp = mamba1_inputs(seed=l, b=b, d=d, l=l, n=n, h0=True)
    rng = np.random.default_rng(l)
    raw = (rng.standard_normal((b, d, l)) - 2.0).astype(np.float32)
    bias = (0.5 * rng.standard_normal(d)).astype(np.float32)
    t = {k: torch.from_numpy(np.ascontiguousarray(v)).cuda() for k, v in inp.items()}
    if ws is not None:
        real = _lib.lib()
        per = 4 * 17 * b * d

        class Limited:
            def __getattr__(self, name):
                if name == "mamba1_scan_workspace_size":
                    return lambda a: min(ws * per, real.mamba1_scan_workspace_size(a))
                return getattr(real, name)

        monkeypatch.setattr(_lib, "lib", Limited)
    state = t["h0"].clone()  # read and written by the same call
    y, hT = mamba_hip.mamba1_scan(t["u"], torch.from_numpy(raw).cuda(), t["A"], t["B"], t["C"], t["D"],
                                  t["z"] if gate else None, delta_bias=torch.from_numpy(bias).cuda(),
                                  delta_softplus=True, initial_state=state, final_state=state)
    torch.cuda.synchronize()
    yr, hr = oracle.mamba1_scan(inp["u"], raw, inp["A"], inp["B"], inp["C"], inp["D"], inp["z"] if gate else None,
                                delta_bias=bias, delta_softplus=True, h0=inp["h0"])
    np.testing.assert_allclose(y.cpu().numpy(), yr, **TOL)
    np.testing.assert_allclose(hT.cpu().numpy(), hr, **TOL)
    assert hT.data_ptr() == state.data_ptr()


# rows at odd addresses on both sides of the rule between the two tiled kernels:
# last half-tiles up to 48 tokens, and up to 80 where the launch is large
@pytest.mark.parametrize("b,d,l", [(2, 70, 1), (2, 70, 15), (2, 70, 17), (1, 70, 33), (1, 70, 47), (1, 70, 49),
                                   (1, 70, 65), (8, 4100, 49), (8, 4100, 65), (8, 4100, 79), (8, 4100, 81)])
def test_odd_rows_match_oracle(b, d, l):
    import torch
    import mamba_hip
    import oracle
    inp = mamba1_inputs(seed=l, b=b, d=d, l=l, n=16, h0=True)
    t = {k: torch.from_numpy(np.ascontiguousarray(v)).cuda() for k, v in inp.items()}
    y, hT = mamba_hip.mamba1_scan(t["u"], t["delta"], t["A"], t["B"], t["C"], t["D"], initial_state=t["h0"])
    torch.cuda.synchronize()
    yr, hr = oracle.mamba1_scan(inp["u"], inp["delta"], inp["A"], inp["B"], inp["C"], inp["D"], h0=inp["h0"])
    np.testing.assert_allclose(y.cpu().numpy(), yr, **TOL)
    np.testing.assert_allclose(hT.cpu().numpy(), hr, **TOL)
