"""The native packing library belongs to the torch it was built against: any
other pairing is a G950Error that names the remedy, not an ImportError."""
import pytest

torch = pytest.importorskip("torch")

from compiler_amd import runtime as rt  # noqa: E402


def test_packer_loads_with_its_own_torch(monkeypatch):
    monkeypatch.setattr(rt, "_packer", None)
    assert torch.__version__.startswith(rt._load_packer().torch_version)


def test_packer_of_another_torch_is_a_g950_error(monkeypatch, tmp_path):
    monkeypatch.setattr(rt, "_packer", None)
    monkeypatch.setattr(torch, "__version__", "1.13.0")
    with pytest.raises(rt.G950Error, match="built against torch"):
        rt._load_packer()
    broken = tmp_path / "g950_py.so"
    broken.write_bytes(b"not a library of this torch")
    monkeypatch.setattr(rt, "PYLIB_PATH", broken)
    with pytest.raises(rt.G950Error, match="does not load with torch") as e:
        rt._load_packer()
    assert e.value.code == rt.RESOURCE
    monkeypatch.setattr(rt, "PYLIB_PATH", tmp_path / "missing.so")
    with pytest.raises(rt.G950Error, match="not built"):
        rt._load_packer()
