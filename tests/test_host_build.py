"""The build leaves out a back-end option that the compiler does not know."""
import os

import pytest

from pdl_amd import build as B

pytestmark = pytest.mark.skipif(not os.path.exists(B.HIPCC), reason="no hipcc")


def extra():
    return {name: flags for _, name, flags in B.units()}


def test_known_options():
    assert B.known([]) and not B.known(["-mllvm", "-amdgpu-no-such-option=1"])
    assert extra()["tile"] == (B.VGPR_FORM if B.known(B.VGPR_FORM) else [])


def test_unknown_option_is_left_out(monkeypatch):
    monkeypatch.setattr(B, "VGPR_FORM", ["-mllvm", "-amdgpu-no-such-option=1"])
    assert all(extra()[name] == [] for name in ("tile", "hgemm", "batch"))
