"""The rounds that a solve reports: the same number whether the short rounds run
as launches of their own or in one workgroup."""
import os
import subprocess
import sys

import pytest

from tests.emu import emu
from tests.test_crowded_cells import TINY
from tests.test_round_routes import ROOT, SMALL


def counts(lib, case, seed):
    code = ("from tests import test_long_segments as t; from tests.emu import emu; "
            f"_, _, st = emu.solve(*t.segments(*{case!r})); "
            "print('COUNTS', {k: st[k] for k in ('insert_rounds', 'flip_rounds', 'flips', 'constraint_rounds', 'segments')})")
    env = dict(os.environ, EMU_SEED=str(seed), EMU_CONC="8", EMU_LIB=lib)
    r = subprocess.run([sys.executable, "-c", code], cwd=ROOT, env=env, capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-3000:]
    return [line for line in r.stdout.splitlines() if line.startswith("COUNTS")]


@pytest.mark.parametrize("case", [("rows", 3000, 25), ("columns", 1200, 10), ("steep", 5000, 40)], ids=lambda c: c[0])
def test_counts_do_not_depend_on_the_route(case):
    whole = counts(emu.build(TINY), case, 1)
    assert counts(emu.build(), case, 2) == whole
    assert counts(emu.build(SMALL), case, 3) == whole
