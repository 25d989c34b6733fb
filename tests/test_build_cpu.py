"""stblarge_amd.build without compiling: which commands it runs, and what it leaves when one of them fails."""

import os
import stat
import subprocess

import pytest

from stblarge_amd import build


def _script(path, text):
    path.write_text("#!/bin/sh\n" + text)
    path.chmod(path.stat().st_mode | stat.S_IXUSR)
    return str(path)


@pytest.mark.parametrize("form", ["bare name", "path"])
def test_binding_finds_the_rocm_headers_whatever_the_form_of_hipcc(monkeypatch, form):
    monkeypatch.setattr(build, "HIPCC", "hipcc" if form == "bare name" else "/opt/rocm/bin/hipcc")
    monkeypatch.setenv("PATH", "/opt/rocm/bin:" + os.environ["PATH"])
    monkeypatch.delenv("ROCM_PATH", raising=False)
    cmd = build.bind_command("out.so")
    dirs = [cmd[i + 1] for i, c in enumerate(cmd) if c == "-isystem"]
    assert all(os.path.isabs(d) for d in dirs), dirs
    assert any(os.path.exists(os.path.join(d, "hip", "hip_runtime_api.h")) for d in dirs), dirs


def _fake(monkeypatch, tmp_path, lib_script, bind_command):
    monkeypatch.setattr(build, "HIPCC", _script(tmp_path / "hipcc", lib_script))
    monkeypatch.setattr(build, "LIB", str(tmp_path / "lib.so"))
    monkeypatch.setattr(build, "BIND", str(tmp_path / "bind.so"))
    monkeypatch.setattr(build, "bind_command", bind_command)


WRITE_LAST = 'for a in "$@"; do out=$a; done; echo new > "$out"\n'  # the output is the last argument


@pytest.mark.parametrize("why", ["no compiler", "no torch", "compile error"])
def test_build_without_the_binding_still_gives_the_library(monkeypatch, tmp_path, capfd, why):
    def command(out):
        if why == "no torch":
            raise ImportError("No module named 'torch'")
        return [str(tmp_path / "absent")] if why == "no compiler" else ["false"]

    _fake(monkeypatch, tmp_path, "sleep 0.2\n" + WRITE_LAST, command)
    (tmp_path / "bind.so").write_text("old")
    assert build.build() == str(tmp_path / "lib.so")
    assert (tmp_path / "lib.so").read_text() == "new\n"
    assert not (tmp_path / "bind.so").exists()  # the old one may not fit the new library
    assert "bind.so" in capfd.readouterr().err


def test_a_failed_library_leaves_no_compiler_running(monkeypatch, tmp_path):
    started = []
    popen = subprocess.Popen

    def record(*a, **k):
        started.append(popen(*a, **k))
        return started[-1]

    _fake(monkeypatch, tmp_path, "exit 1\n", lambda out: ["sh", "-c", f"sleep 2; echo new > {out}"])
    monkeypatch.setattr(subprocess, "Popen", record)
    (tmp_path / "lib.so").write_text("old")
    with pytest.raises(subprocess.CalledProcessError):
        build.build()
    assert started and all(p.poll() is not None for p in started)
    assert (tmp_path / "lib.so").read_text() == "old"
