"""Tiles of the pseudopotential triplets around a wavefront's window of 64
segments per atom, and PP lists built without the structure's own lists.  Lists
and blocks equal the oracle's."""
import numpy as np
import pytest

import oracle
from fireball_hip import synth
from fireball_hip.lib import Assembler
from golden.make_golden import PP_LIST_KEYS

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 64, 65, 66, 67])
def test_segments_around_a_window(n):
    sp = synth.with_pp([synth.SI])
    ts = synth.add_pp_tables(synth.make_tables(sp))
    rng = np.random.default_rng(5)
    pos = []
    while len(pos) < n:
        p = rng.uniform(-1.6, 1.6, 3)
        if p @ p < 2.56 and all(np.linalg.norm(p - q) > 0.55 for q in pos):
            pos.append(p)
    st = synth.Structure(np.array(pos) + 20.0, np.ones(n, np.int32), np.diag([40.0] * 3), 1)
    o = oracle.System(oracle.Tables(ts), st)
    o.build_lists()
    ref = o.run_pp()
    asm = Assembler(ts, precision="fp64")
    asm.add_structure(st)
    asm.build_lists_pp()      # bins the atoms itself
    first = asm.pp_lists()
    asm.build_lists()
    asm.build_lists_pp()
    asm.assemble_pp()
    again = asm.pp_lists()
    for k in PP_LIST_KEYS:
        assert np.array_equal(first[k], ref[k]) and np.array_equal(again[k], ref[k]), k
    for k in ("SVNL", "VNL"):
        assert np.array_equal(asm.pp_blocks(k), ref[k]), k
    asm.close()
