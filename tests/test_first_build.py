"""The build entry from a checkout that holds no built file, in one process.

The package is imported before its libraries exist (the build lives in it), so what the import
found must not decide what the build's own process can load afterwards. The compilers are
stand-ins that deliver this tree's built files; the order of import, build and first use is
that of the build entry."""
import os
import shutil
import subprocess
import sys

import pytest

from kvq_decode_amd import _lib

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ENTRY = """
import warnings
with warnings.catch_warnings(record=True) as seen:
    warnings.simplefilter("always")
    import __graft_entry__
    __graft_entry__.build()
    from kvq_decode_amd import _lib, ops
    print("version", _lib.version())
    print("host", getattr(_lib.host, "__file__", None))
    print("warned", [str(w.message) for w in seen if "_host.so" in str(w.message)])
"""


def _checkout(tmp, host):
    """The sources without any built file, and compilers that write `host` and this tree's
    libkvq.so where a compiler would (objects: empty files)."""
    root = tmp / "checkout"
    shutil.copytree(os.path.join(REPO, "kvq_decode_amd"), root / "kvq_decode_amd",
                    ignore=shutil.ignore_patterns("*.so", "_build", "__pycache__"))
    shutil.copytree(os.path.join(REPO, "include"), root / "include")
    shutil.copy(os.path.join(REPO, "__graft_entry__.py"), root)
    env = dict(os.environ, PYTHONPATH=str(root))
    for var, built in (("HIPCC", _lib.LIB_PATH), ("CXX", host)):
        script = tmp / var.lower()
        script.write_text('#!/bin/sh\nfrom=' + f'"{built}"' + '\n'
                          'while [ "$1" != "-o" ]; do [ "$1" = "-c" ] && from=/dev/null; shift; done\n'
                          'exec cp "$from" "$2"\n')
        script.chmod(0o755)
        env[var] = str(script)
    return root, env


def _build(root, env):
    r = subprocess.run([sys.executable, "-c", ENTRY], cwd=root, env=env, capture_output=True,
                       text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    return r.stdout


def test_build_then_use_in_one_process(tmp_path):
    """A first build's own process loads both libraries it built, and so does the next one's,
    which finds them there before it builds."""
    root, env = _checkout(tmp_path, os.path.join(REPO, "kvq_decode_amd", "_host.so"))
    for _ in range(2):
        out = _build(root, env)
        assert f"host {root / 'kvq_decode_amd' / '_host.so'}" in out
        assert "warned []" in out


@pytest.mark.parametrize("broken", ["no compiler", "no module"])
def test_build_without_the_native_host_path(tmp_path, broken):
    """Without a C++ compiler, or with a module that does not load, the library still works,
    and a warning says why calls take the Python path."""
    bad = tmp_path / "bad.so"
    bad.write_bytes(b"no shared object")
    root, env = _checkout(tmp_path, bad)
    if broken == "no compiler":
        env["CXX"] = str(tmp_path / "missing")
    out = _build(root, env)
    assert "version kvq" in out and "host None" in out
    assert ("not found" if broken == "no compiler" else "does not load") in out


def test_cu_counts_reach_a_host_path_loaded_later(monkeypatch):
    """A device's compute units, asked for before the library is loaded, are passed on."""
    told = []

    class Module:
        @staticmethod
        def bind(*args):
            pass

        @staticmethod
        def set_cu_count(device, count):
            told.append((device, count))

    L = _lib.lib()
    monkeypatch.setattr(_lib, "host", _lib._NoHost)
    monkeypatch.setattr(_lib, "_cu_counts", {})
    monkeypatch.setattr(_lib.importlib, "import_module", lambda name: Module)
    _lib.set_cu_count(3, 256)
    assert told == []
    _lib._load_host(L)
    assert _lib.host is Module and told == [(3, 256)]
    _lib.set_cu_count(1, 304)
    assert told == [(3, 256), (1, 304)]
