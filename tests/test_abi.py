"""The C-ABI library loads on a machine without a GPU and exports every
symbol that include/*.h declares (no compute calls are made here)."""

import ctypes
import re
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]


def declared():
    names = set()
    for h in (ROOT / "include").glob("*.h"):
        text = h.read_text()
        text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
        names.update(re.findall(r"\b(hk_\w+)\s*\(", text))
    return sorted(names)


def test_header_declares_symbols():
    assert "hk_mlstm_step" in declared()


def test_library_exports_every_declared_symbol():
    from hackathon_amd import _lib

    if not _lib.LIB_PATH.exists():
        pytest.fail("libhackathon_amd.so is not built (run __graft_entry__.build())")
    handle = ctypes.CDLL(str(_lib.LIB_PATH))
    missing = [n for n in declared() if not hasattr(handle, n)]
    assert not missing, f"not exported: {missing}"


def test_python_binding_covers_header():
    from hackathon_amd import _lib
    import hackathon_amd.engine  # noqa: F401  (registers the engine signatures)
    import hackathon_amd.weights  # noqa: F401  (registers the host-side helpers)

    assert set(declared()) <= set(_lib.declared_symbols())
    lib = _lib.lib()
    assert lib.hk_version() >= 1
    assert isinstance(lib.hk_last_error(), bytes)


@pytest.mark.parametrize("raw", [True, False])
def test_current_stream_takes_what_torch_takes(monkeypatch, raw):
    """_lib.current_stream on a device, its name, its index and a device
    without an index, with and without torch's raw-handle binding (stubs: no
    GPU here)."""
    import torch
    from types import SimpleNamespace

    from hackathon_amd import _lib

    monkeypatch.setattr(torch.cuda, "current_stream", lambda d: SimpleNamespace(cuda_stream=41))
    if raw:
        monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda i: 42 + i, raising=False)
    else:
        monkeypatch.delattr(torch._C, "_cuda_getCurrentRawStream", raising=False)
    assert _lib.current_stream(torch.device("cuda:1")) == (43 if raw else 41)
    for device in (torch.device("cuda"), "cuda:0", 0, None):
        assert _lib.current_stream(device) == 41
