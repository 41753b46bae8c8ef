"""The units of the build can be listed where there is no compiler."""
from pdl_amd import build as B


def test_units_without_a_compiler(monkeypatch):
    monkeypatch.setattr(B, "HIPCC", "/nonexistent/hipcc")
    assert not B.known([])
    assert "tile" in [name for _, name, _ in B.units()]
