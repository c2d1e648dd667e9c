"""Tiles of the pseudopotential triplets around a wavefront's window of 64
segments per atom, and PP lists built without the structure's own lists.  Lists
and blocks equal the oracle's."""
import ctypes as C

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


def test_longer_cutoffs_on_structures_that_are_on_the_gpu():
    """fb_set_species between two PP list builds: the second equals a fresh context's."""
    sp = synth.with_pp([synth.SI])
    ts = synth.add_pp_tables(synth.make_tables(sp))
    st = synth.diamond_si((4, 4, 4), sigma=0.05, seed=2)

    def cutoffs(asm, scale):
        nssh, lssh = np.array([2], np.int32), np.array([[0, 1, 0, 0]], np.int32)
        rc = scale * np.array([[*sp[0].rcutoffA, 0.0, 0.0]])
        asm._check(asm.L.fb_set_species(asm.h, 1, None, nssh.ctypes.data_as(C.POINTER(C.c_int)),
                                        lssh.ctypes.data_as(C.POINTER(C.c_int)),
                                        rc.ctypes.data_as(C.POINTER(C.c_double))))
        asm._check(asm.L.fb_commit_tables(asm.h))

    fresh = Assembler(ts, precision="fp64")
    fresh.add_structure(st)
    fresh.build_lists_pp()
    want = fresh.pp_lists()
    asm = Assembler(ts, precision="fp64")
    cutoffs(asm, 0.6)
    asm.add_structure(st)
    asm.build_lists_pp()
    assert not np.array_equal(asm.pp_lists()["pp_n"], want["pp_n"])
    cutoffs(asm, 1.0)
    asm.build_lists_pp()
    got = asm.pp_lists()
    for k in PP_LIST_KEYS:
        assert np.array_equal(got[k], want[k]), k
    asm.close()
    fresh.close()


def test_cells_after_a_list_build_that_failed():
    """Wider PP cutoffs on the GPU, a PP list build refused under capture, then the same build outside."""
    sp = synth.with_pp([synth.SI])
    ts = synth.add_pp_tables(synth.make_tables(sp))
    st = synth.diamond_si((4, 4, 4), sigma=0.05, seed=2)

    def pp_cutoff(asm, rc):
        npp, lpp, clv = np.array([2], np.int32), np.array([[0, 1, 0, 0]], np.int32), np.array([[-2.6, 1.3, 0.0, 0.0]])
        rpp = np.array([rc])
        asm._check(asm.L.fb_set_species_pp(asm.h, npp.ctypes.data_as(C.POINTER(C.c_int)),
                                           lpp.ctypes.data_as(C.POINTER(C.c_int)),
                                           rpp.ctypes.data_as(C.POINTER(C.c_double)),
                                           clv.ctypes.data_as(C.POINTER(C.c_double))))
        asm._check(asm.L.fb_commit_tables(asm.h))

    fresh = Assembler(ts, precision="fp64")
    pp_cutoff(fresh, 4.0)
    fresh.add_structure(st)
    fresh.build_lists_pp()
    want = fresh.pp_lists()
    hip = C.CDLL("libamdhip64.so")
    stream, graph = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreateWithFlags(C.byref(stream), C.c_uint(1)) == 0
    asm = Assembler(ts, precision="fp64")
    asm._check(asm.L.fb_set_stream(asm.h, stream))
    asm.add_structure(st)
    asm.build_lists()
    pp_cutoff(asm, 4.0)
    asm.assemble_all()   # sends the structures
    assert hip.hipStreamBeginCapture(stream, C.c_int(1)) == 0
    try:
        n = C.c_int64()
        assert asm.L.fb_build_lists_pp(asm.h, C.byref(n), C.byref(n), C.byref(n)) != 0
    finally:
        hip.hipStreamEndCapture(stream, C.byref(graph))
        if graph.value:
            hip.hipGraphDestroy(graph)
    hip.hipGetLastError()
    asm._check(asm.L.fb_set_stream(asm.h, None))   # the capture's stream stays invalid
    asm.build_lists_pp()
    got = asm.pp_lists()
    for k in PP_LIST_KEYS:
        assert np.array_equal(got[k], want[k]), k
    asm.close()
    fresh.close()
