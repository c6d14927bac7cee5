"""The build of the host layers, with the compiler calls recorded instead of run."""
import sys

from nanoinfer_amd import build as nb


def _artifacts(monkeypatch):
    cmds = []
    monkeypatch.setattr(nb, "_run", lambda cmd, what: cmds.append(what))
    monkeypatch.setattr(nb.os, "replace", lambda a, b: None)
    return nb._host_artifacts(), cmds


def test_host_layers_build_without_torch(monkeypatch):
    monkeypatch.setitem(sys.modules, "torch", None)  # import torch raises ImportError
    out, cmds = _artifacts(monkeypatch)
    assert nb.HOST_LIB in out and nb.HOST_TEST in out and any("nicpp" in p for p in out)
    assert not any("_calls" in p for p in out) and "_calls module" not in cmds


def test_calls_build_last(monkeypatch):
    out, cmds = _artifacts(monkeypatch)
    assert "_calls" in out[-1] and cmds[-1] == "_calls module" and len(out) == 4
