"""The prefill conv at every tile length its launch takes (8 to 64 positions per
workgroup) and every kernel length whose margin to the second tile differs,
ragged ends and sequences shorter than the window, with the window updated in
place by the first tile's workgroups, vs the oracle (f32: rtol 1e-4; the window
holds input values: exact)."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# (b, l, channels): tiles of 64 (twice), 32 and 8 positions; scalar channels; l < kernel
CASES = [(8, 4101, 8), (4, 4101, 8), (2, 4101, 8), (1, 500, 16), (2, 300, 7), (3, 2, 24), (1, 1, 8)]
# tiles of 32, 16 (the first of 8 positions) and 8, where a kernel of 8 leaves the
# second tile one position past the old window
KERNELS = [(2, 4101, 8), (1, 4101, 8), (1, 500, 16), (1, 4101, 7)]


@pytest.mark.parametrize("case", CASES)
def test_conv1d_fwd(case):
    _check(*case, 4)


@pytest.mark.parametrize("K", [2, 4, 8])
@pytest.mark.parametrize("case", KERNELS)
def test_conv1d_fwd_kernels(case, K):
    _check(*case, K)


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("K", [1, 2, 3, 4, 8])
@pytest.mark.parametrize("l,c", [(1, 16), (3, 16), (4, 7), (7, 16), (8, 24), (9, 16), (15, 7)])
def test_conv1d_fwd_of_one_tile(l, c, K, off):
    """At most 8 positions: the new window is what slid through the old one, on both
    sides of the kernel's length; whole rows of weights and window where they are
    16-byte aligned (off 0, kernels of 4 and 8), a word at a time elsewhere."""
    _check(2, l, c, K, off)


def _check(b, L, c, K, off=0):
    import torch
    import mamba_hip
    import oracle
    rng = np.random.default_rng(b + L + c)
    x, st = rng.standard_normal((b, L, c), dtype=np.float32), rng.standard_normal((b, c, K), dtype=np.float32)
    w, bias = rng.standard_normal((c, K), dtype=np.float32), rng.standard_normal(c, dtype=np.float32)
    g = lambda a: torch.from_numpy(a).cuda()  # noqa: E731
    s = torch.empty(st.size + off, device="cuda")[off:].view(st.shape).copy_(g(st))
    out = mamba_hip.conv1d_fwd(g(x), s, g(w), g(bias))
    torch.cuda.synchronize()
    want, _, wst = oracle.mamba2_conv_fwd(x, w, bias, st, np.zeros(0), 0, 0, c, 0)
    np.testing.assert_allclose(out.cpu().numpy(), want, rtol=1e-4, atol=2e-5)
    np.testing.assert_array_equal(s.cpu().numpy(), wst.astype(np.float32))
