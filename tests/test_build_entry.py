"""build() compiles the reference-based harness only where the reference's sources are: an empty
folder in their place is no error."""
import subprocess

import __graft_entry__ as entry


def _commands(monkeypatch, ref):
    ran = []
    monkeypatch.setattr(subprocess, "run", lambda cmd, **kw: ran.append(cmd))
    monkeypatch.setenv("CRUCIBLE_REF", str(ref))
    entry.build()
    return ran


def test_reference_harness_only_with_its_sources(monkeypatch, tmp_path):
    assert not any("ref" in cmd for cmd in _commands(monkeypatch, tmp_path))
    assert not any("ref" in cmd for cmd in _commands(monkeypatch, tmp_path / "absent"))
    header = tmp_path / "engine/exl3/kernels/lane_window.h"
    header.parent.mkdir(parents=True)
    header.write_text("")
    assert any("ref" in cmd and f"REF={tmp_path}" in cmd for cmd in _commands(monkeypatch, tmp_path))
