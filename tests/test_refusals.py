"""Calls that hand raw pointers to a kernel refuse sizes, types and devices that
do not fit together before anything is launched, as the torch products in their
place do.  On the CPU, with a library of which only the size queries answer."""

import pytest
import torch

import mamba_hip
from mamba_hip import _lib
from mamba_hip.mamba1 import _mm_f32_takes, mm_f32
from mamba_hip.step import linear_row


@pytest.fixture(autouse=True)
def no_launch(monkeypatch):
    real = _lib.lib()

    class Sizes:
        def __getattr__(self, name):
            if name.endswith("_size"):
                return getattr(real, name)
            raise AssertionError(f"reached {name}")
    monkeypatch.setattr(_lib, "lib", Sizes)


MM = [((1, 4, 8), (1, 7, 5), None, "shapes"), ((2, 4, 8), (1, 8, 5), None, "shapes"), ((1, 4, 8), (8, 5), None, "shapes"),
      ((1, 4, 8), (1, 8, 5), (1, 4, 6), "shapes"), ((1, 4, 8), (1, 8, 5), (1, 5, 5), "shapes"),
      ((1, 4, 8), (1, 8, 5), None, "device")]


@pytest.mark.parametrize("a,b,out,what", MM)
def test_mm_f32(a, b, out, what):
    with pytest.raises(mamba_hip.MambaHipError, match=what):
        mm_f32(torch.zeros(a), torch.zeros(b), None if out is None else torch.zeros(out))


def test_mm_f32_types_and_rows_of_out():
    a, b = torch.zeros(1, 4, 8), torch.zeros(1, 8, 5)
    with pytest.raises(mamba_hip.MambaHipError, match="float32|device"):
        mm_f32(a, b.double())
    with pytest.raises(mamba_hip.MambaHipError, match="out"):
        mm_f32(a, b, torch.zeros(1, 4, 10)[:, :, ::2])


def test_the_library_keeps_empty_and_autocast_products():
    a, b = torch.zeros(4, 8), torch.zeros(8, 5)
    assert _mm_f32_takes(a, b)
    assert not _mm_f32_takes(a[:0], b)  # no rows: an empty product, not an error
    torch.set_autocast_enabled("cuda", True)
    try:
        assert not _mm_f32_takes(a, b)
    finally:
        torch.set_autocast_enabled("cuda", False)


def test_mamba1_forward_width():
    m = mamba_hip.Mamba1Config(64).init("cpu")
    cache = m.new_cache(2)
    with pytest.raises(RuntimeError, match="shapes"):
        m.forward(torch.zeros(2, 16, 80), cache)
    assert not cache.conv_bik.any() and not cache.ssm_bir.any()


def test_linear_row():
    f, bf = torch.float32, torch.bfloat16
    t = lambda n, dtype=f: torch.zeros(n, dtype=dtype)  # noqa: E731
    packed = t(_lib.lib().mamba_linear_packed_size(64, 96), torch.uint8)
    for x, w, out, norm, bias in [(t(80, bf), packed, t(96), None, None), (t(64, bf), packed, t(128), None, None),
                                  (t(64), packed, t(96), t(48), None), (t(64), packed, t(96), t(64, bf), None),
                                  (t(64, bf), packed, t(96), None, t(64)), (t(128, bf)[::2], packed, t(96), None, None)]:
        with pytest.raises(mamba_hip.MambaHipError, match="linear_row"):
            linear_row(x, w, out, norm_w=norm, bias=bias)


@pytest.mark.parametrize("b", [1, 2])
def test_mamba3_stack_width(b, monkeypatch):
    monkeypatch.setattr("mamba_hip.mamba3.packed_weight", lambda w: torch.zeros(1, dtype=torch.uint8))
    stack = mamba_hip.Mamba3Stack.init(mamba_hip.Mamba3Config(64, state_rank=32), 2, "cpu")
    with pytest.raises(mamba_hip.MambaHipError, match="d_model"):
        stack.step_(torch.zeros(b, 128), stack.new_caches(b))
