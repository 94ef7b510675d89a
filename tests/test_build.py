"""The build leaves either libraries of the present sources or none."""
import pytest

from embla_attn import build as b


def fake_tree(tmp_path, monkeypatch, hipcc):
    """build's paths moved under tmp_path, an older build's libraries there, hipcc a shell script."""
    (tmp_path / "csrc").mkdir()
    (tmp_path / "csrc" / "a.hip").write_text("int x;\n")
    exe = tmp_path / "hipcc"
    exe.write_text("#!/bin/sh\n" + hipcc)
    exe.chmod(0o755)
    libs = {}
    for name in ("LIB", "HOST_LIB", "PROBE_LIB"):
        libs[name] = tmp_path / f"{name}.so"
        libs[name].write_text("older")
        monkeypatch.setattr(b, name, libs[name])
    monkeypatch.setattr(b, "CSRC", tmp_path / "csrc")
    monkeypatch.setattr(b, "OBJ", tmp_path / "_build")
    monkeypatch.setattr(b, "HIPCC", str(exe))
    return libs


# a compile that fails; compiles that pass and a link that fails
@pytest.mark.parametrize("hipcc, message", [("exit 1\n", "hipcc failed on a.hip"),
                                            ('case "$*" in *-shared*) exit 1;; esac\n', "link failed")])
def test_a_failed_build_leaves_no_older_library(tmp_path, monkeypatch, hipcc, message):
    libs = fake_tree(tmp_path, monkeypatch, hipcc)
    with pytest.raises(RuntimeError, match=message):
        b.build()
    assert not any(p.exists() for p in libs.values())
