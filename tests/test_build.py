"""The build: the library stands without the test infrastructure, and its sources
ask no compiler builtin of the CPU stand-in for the HIP runtime that a
stand-in without scoped read-modify-write atomics has not got."""
import os
import re
import subprocess

import pytest

import __graft_entry__ as entry
from tests.emu import build_emu

SCOPED = re.compile(r"template <class T, class V>\s*inline T __hip_atomic_fetch_\w+\(.*?\n}\n", re.S)


@pytest.mark.parametrize("source", ["mesh.hip", "cons.hip", "steiner.hip"])
def test_sources_need_no_scoped_atomics_of_the_stand_in(source, tmp_path):
    (tmp_path / "hip").mkdir()
    with open(os.path.join(build_emu.HERE, "hip", "hip_runtime.h")) as f:
        stand_in = SCOPED.sub("", f.read())
    assert "__hip_atomic_fetch_" not in stand_in
    (tmp_path / "hip" / "hip_runtime.h").write_text(stand_in)
    for name in build_emu.HEADERS + [source]:
        with open(os.path.join(build_emu.CSRC, name)) as f:
            txt = f.read().replace('"../../include/', f'"{build_emu.ROOT}/include/')
        (tmp_path / name).write_text(build_emu.rewrite_shared(build_emu.rewrite_launches(txt)))
    r = subprocess.run([build_emu.CXX, "-std=c++17", "-fsyntax-only", "-Wno-attributes", "-Wno-unknown-pragmas",
                        "-I", str(tmp_path), "-x", "c++", str(tmp_path / source)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]


def test_library_is_built_and_loaded_before_the_test_builds(monkeypatch):
    import gcdt_amd
    from gcdt_amd import build as product
    from oracle import oracle
    from tests import host_bodies

    done = []

    def broken():
        raise RuntimeError("test infrastructure does not build")
    monkeypatch.setattr(product, "build", lambda verbose=False: done.append("built"))
    monkeypatch.setattr(gcdt_amd, "lib", lambda: done.append("loaded"))
    monkeypatch.setattr(oracle, "build", broken)
    monkeypatch.setattr(host_bodies, "build", broken)
    with pytest.raises(RuntimeError):
        entry.build()
    assert done == ["built", "loaded"]
