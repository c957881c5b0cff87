"""The compile recipes: a compiler that fails ends the build, also where it
has written its output, and the failing command is printed."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def make(tmp_path, where, status, *args):
    cc = tmp_path / "compiler"
    cc.write_text('#!/bin/sh\nout=\nwhile [ $# -gt 0 ]; do [ "$1" = -o ] && out=$2; shift; done\n'
                  'echo x > "$out"; echo "a diagnostic" >&2; exit %d\n' % status)
    cc.chmod(0o755)
    return subprocess.run(["make", "-s", "-C", os.path.join(ROOT, where), f"HIPCC={cc}", *args],
                          capture_output=True, text=True, timeout=60)


@pytest.mark.parametrize("status", [0, 3])
def test_the_compilers_status_is_the_builds(tmp_path, status):
    out = tmp_path / "lib.so"
    r = make(tmp_path, "hachiue_amd/csrc", status, f"OBJ={tmp_path}/obj", f"OUT={out}")
    assert (r.returncode != 0) == (status != 0)
    assert out.exists() == (status == 0)
    assert "a diagnostic" in r.stderr
    if status:
        assert f"exit status 3: {tmp_path}/compiler" in r.stderr


def test_the_sanitizer_builds_too(tmp_path):
    os.mkdir(tmp_path / "san")
    r = make(tmp_path, "tests/sanitize", 3, f"OUT={tmp_path}/san", f"{tmp_path}/san/capi_asan.o")
    assert r.returncode != 0 and "exit status 3" in r.stderr
    assert not (tmp_path / "san" / "capi_asan.o").exists()
