"""The native call module and the library it calls (no GPU needed)."""
from __future__ import annotations

import shutil
import subprocess
import sys

from engine.kernels import _native


def _run(code: str, folder) -> str:
    """Runs code in a process of its own, with _native's library looked for in folder."""
    setup = ("import sys; sys.path.insert(0, {pkg!r}); import torch\n"
             "from engine.kernels import _native\n"
             "_native.LIB_PATH = _native.Path({lib!r})\n")
    pkg = str(_native.LIB_PATH.parents[2])
    done = subprocess.run([sys.executable, "-c",
                           setup.format(pkg=pkg, lib=str(folder / "another.so")) + code],
                          capture_output=True, text=True, timeout=300)
    assert done.returncode == 0, done.stderr
    return done.stdout


def test_the_module_calls_the_library_that_is_loaded(tmp_path):
    """Another build of the library, opened under its own name, is the only one in the process."""
    shutil.copy(_native.LIB_PATH, tmp_path / "another.so")
    shutil.copy(_native.LIB_PATH.with_name("_pa_host.so"), tmp_path / "_pa_host.so")
    out = _run("m = _native.host()\n"
               "maps = open('/proc/self/maps').read()\n"
               "print('another.so' in maps, '_pa_host.so' in maps, 'libpa_gfx950.so' in maps)\n"
               "print(len(m.CALLS))", tmp_path)
    assert out.split() == ["True", "True", "False", "5"]


def test_a_stale_module_is_refused(tmp_path):
    """Built before the library's interface last changed: refused as a stale library is."""
    shutil.copy(_native.LIB_PATH, tmp_path / "another.so")
    shutil.copy(_native.LIB_PATH.with_name("_pa_host.so"), tmp_path / "_pa_host.so")
    out = _run("_native.load()\n"
               "_native.ABI_VERSION += 1\n"
               "try:\n"
               "    _native.host()\n"
               "except _native.NativeLibraryError as e:\n"
               "    print(e)", tmp_path)
    assert f"_pa_host.so has ABI {_native.ABI_VERSION}, the bindings expect" in out
