"""CPU: which objects an incremental build takes as current."""

from __future__ import annotations

import os

from cugo_amd import build


def test_objects_older_than_the_flags_are_compiled_again(tmp_path, monkeypatch):
    """The compile flags are in build.py, so an object older than it may have been built with
    others: build_library(force=False) compiles it again, and only then."""
    names = build.SOURCES
    (tmp_path / "csrc").mkdir()
    (tmp_path / "_build").mkdir()
    script = tmp_path / "build.py"
    for f in (script, tmp_path / "header", tmp_path / "csrc" / "stop_bits.inc",
              *(tmp_path / "csrc" / n for n in names), *(tmp_path / "_build" / f"{n}.o" for n in names),
              tmp_path / "libcugo_hip.so"):
        f.write_text("")
        os.utime(f, (1000, 1000))
    compiled = []

    class Done:
        def __init__(self, cmd):
            compiled.append(cmd)

        def wait(self):
            return 0

    monkeypatch.setattr(build, "PKG", tmp_path)
    monkeypatch.setattr(build, "CSRC", tmp_path / "csrc")
    monkeypatch.setattr(build, "HEADERS", (tmp_path / "header",))
    monkeypatch.setattr(build, "__file__", str(script))
    monkeypatch.setattr(build, "generate_stop_bits", lambda force: None)
    monkeypatch.setattr(build, "_run", lambda cmd: None)
    monkeypatch.setattr(build, "check_no_packed_fp32", lambda lib: None)
    monkeypatch.setattr(build.subprocess, "Popen", Done)
    build.build_library(force=False)
    assert not compiled
    os.utime(script, (2000, 2000))
    build.build_library(force=False)
    assert len(compiled) == len(names)
