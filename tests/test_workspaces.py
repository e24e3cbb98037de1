"""The size queries ask for what the call's kernels use (host arithmetic only: no
GPU; pointers stand for aligned tensors and are not followed)."""

import ctypes

from mamba_hip import _lib

PTR = 1 << 20


def _bwd2(b, l, h, n, g=1, p=64):
    a = _lib.Ssd2BwdArgs()
    a.batch, a.seqlen, a.nheads, a.headdim, a.ngroups, a.dstate = b, l, h, p, g, n
    for k in ("x", "dt", "A", "B", "C", "dy", "dx", "ddt", "dA", "dB", "dC", "d_initial_state"):
        setattr(a, k, PTR)
    for k, w, q in (("x", h * p, p), ("dy", h * p, p), ("B", g * n, n), ("C", g * n, n)):
        setattr(a, f"{k}_sb", l * w)
        setattr(a, f"{k}_sl", w)
        setattr(a, f"{k}_s{'g' if k in 'BC' else 'h'}", q)
    a.dt_sb, a.dt_sl, a.dt_sh = l * h, h, 1
    return a


def test_bf16_backward_asks_for_64_row_entry_states_only():
    """A full chip (one segment): a state per 64 positions, dB and dC per head,
    partial sums.  The f32 query also covers the SIMT kernels' state per 32, which
    a call with other alignments takes."""
    b, l, h, n = 4, 4096, 64, 128
    a, L = _bwd2(b, l, h, n), _lib.lib()
    state, planes, sums = b * h * 64 * n * 4, 2 * b * l * h * n * 4, 2 * -(-b * h * 4 // 256) * 256
    assert L.mamba_ssd2_bwd_bf16_workspace_size(ctypes.byref(a)) == l // 64 * state + planes + sums
    assert L.mamba_ssd2_bwd_workspace_size(ctypes.byref(a)) == l // 32 * state + planes + sums
    assert L.mamba_ssd2_bwd_bf16(ctypes.byref(a), ctypes.c_void_p(PTR), l // 64 * state, None, None, None) == 3  # too small
