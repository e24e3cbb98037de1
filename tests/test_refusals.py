"""Calls that hand raw pointers to a kernel refuse sizes, types and devices that
do not fit together before anything is launched, as the torch products in their
place do.  On the CPU, with a library that fails the test when it is called."""

import pytest
import torch

import mamba_hip
from mamba_hip import _lib
from mamba_hip.mamba1 import mm_f32


@pytest.fixture(autouse=True)
def no_launch(monkeypatch):
    def called():
        raise AssertionError("reached the library")
    monkeypatch.setattr(_lib, "lib", called)


MM = [((1, 4, 8), (1, 7, 5), None, "shapes"), ((2, 4, 8), (1, 8, 5), None, "shapes"), ((1, 4, 8), (8, 5), None, "shapes"),
      ((1, 4, 8), (1, 8, 5), (1, 4, 6), "shapes"), ((1, 4, 8), (1, 8, 5), (1, 5, 5), "shapes"),
      ((1, 4, 8), (1, 8, 5), None, "device")]


@pytest.mark.parametrize("a,b,out,what", MM)
def test_mm_f32(a, b, out, what):
    with pytest.raises(mamba_hip.MambaHipError, match=what):
        mm_f32(torch.zeros(a), torch.zeros(b), None if out is None else torch.zeros(out))


def test_mm_f32_types_and_rows_of_out():
    a, b = torch.zeros(1, 4, 8), torch.zeros(1, 8, 5)
    with pytest.raises(mamba_hip.MambaHipError, match="float32"):
        mm_f32(a, b.double())
    with pytest.raises(mamba_hip.MambaHipError, match="out"):
        mm_f32(a, b, torch.zeros(1, 4, 10)[:, :, ::2])


def test_mamba1_forward_width():
    m = mamba_hip.Mamba1Config(64).init("cpu")
    cache = m.new_cache(2)
    with pytest.raises(RuntimeError, match="shapes"):
        m.forward(torch.zeros(2, 16, 80), cache)
    assert not cache.conv_bik.any() and not cache.ssm_bir.any()
