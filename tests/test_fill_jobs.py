"""FillJobs (mesh.hpp): outputs that were not asked for are left out, and one
fill too many is refused before it is written past the list."""
import os
import subprocess

from tests.emu import build_emu

MAIN = r"""
#include <cstdio>
#include "mesh.hpp"
int main()
{
    int word = 0;
    struct { gcdt::FillJobs f; int after[8]; } s = {};
    s.f.add(nullptr, 7, 5);
    s.f.add(&word, 7, 0);
    if (s.f.njobs != 0) return 1;
    for (int i = 0; i < gcdt::FillJobs::kMax; i++) s.f.add(&word, i, 1);
    if (s.f.njobs != gcdt::FillJobs::kMax) return 2;
    try {
        s.f.add(&word, 9, 1);
    } catch (const gcdt::Error&) {
        for (int a : s.after)
            if (a) return 3;
        return s.f.njobs == gcdt::FillJobs::kMax ? 0 : 4;
    }
    return 5;
}
"""


def test_optional_outputs_and_the_bound(tmp_path):
    for name in build_emu.HEADERS:
        with open(os.path.join(build_emu.CSRC, name)) as f:
            txt = f.read().replace('"../../include/', f'"{build_emu.ROOT}/include/')
        (tmp_path / name).write_text(build_emu.rewrite_shared(build_emu.rewrite_launches(txt)))
    (tmp_path / "main.cpp").write_text(MAIN)
    obj, exe = tmp_path / "main.o", tmp_path / "main"
    flags = [*build_emu.FLAGS, "-I", str(tmp_path)]
    r = subprocess.run([build_emu.CXX, *flags, "-ffunction-sections", "-c", str(tmp_path / "main.cpp"), "-o", str(obj)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([build_emu.CXX, "-Wl,--gc-sections", str(obj), "-o", str(exe), "-lpthread"], capture_output=True,
                       text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    assert subprocess.run([str(exe)]).returncode == 0
