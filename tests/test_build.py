"""CPU: which objects an incremental build makes again."""
import os

from leviathan_amd import build


def test_incremental_build_makes_objects_of_other_flags_again(tmp_path, monkeypatch):
    """An object is kept while its source, the headers and the command that made it are the same."""
    csrc, out = tmp_path / "csrc", tmp_path / "build"
    csrc.mkdir()
    out.mkdir()
    (csrc / "a.hpp").write_text("")
    source = csrc / "a.hip"
    source.write_text("")
    compiler = tmp_path / "hipcc"
    compiler.write_text(f"#!/bin/sh\necho >> {tmp_path}/calls\nwhile [ \"$1\" != -o ]; do shift; done\necho object > \"$2\"\n")
    compiler.chmod(0o755)
    monkeypatch.setattr(build, "CSRC", str(csrc))
    monkeypatch.setattr(build, "OBJ_DIR", str(out))
    monkeypatch.setattr(build, "hipcc", lambda: str(compiler))
    monkeypatch.setattr(build, "_headers_mtime", lambda: os.path.getmtime(csrc / "a.hpp"))

    def calls(extra=(), force=False):
        before = (tmp_path / "calls").read_text().count("\n") if (tmp_path / "calls").exists() else 0
        build._compile(str(source), force, list(extra))
        return (tmp_path / "calls").read_text().count("\n") - before

    assert calls() == 1 and calls() == 0 and calls(force=True) == 1
    monkeypatch.setattr(build, "NO_PRELOAD", {"a.hip"})
    assert calls() == 1 and calls() == 0
    assert calls(["-DX"]) == 1 and calls(["-DX"]) == 0 and calls() == 1
    os.utime(source, (os.path.getmtime(source) + 100,) * 2)
    assert calls() == 1
