"""The build of tritonix_amd/_launch.so: a machine without a compiler for it still gets the library."""
import pytest

from tritonix_amd import build


def test_a_build_without_the_host_compiler_leaves_no_stale_module(monkeypatch, tmp_path):
    (tmp_path / "_launch.so").write_bytes(b"of older sources")
    monkeypatch.setattr(build, "HERE", str(tmp_path))
    monkeypatch.setattr(build, "LIB", str(tmp_path / "lib.so"))
    monkeypatch.setattr(build, "BUILD", str(tmp_path / "build"))
    monkeypatch.setattr(build.subprocess, "run", lambda *_, **__: (_ for _ in ()).throw(FileNotFoundError("g++")))
    monkeypatch.setattr(build, "instance_list", lambda quick: [])
    monkeypatch.setattr(build, "conv_instance_list", lambda quick: [])
    monkeypatch.setattr(build, "_compile", lambda *_: None)
    with pytest.warns(RuntimeWarning, match="_launch.so was not built"), pytest.raises(FileNotFoundError):
        build.build(verbose=False)                           # (the library's own link step needs hipcc)
    assert not (tmp_path / "_launch.so").exists()
