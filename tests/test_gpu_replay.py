"""Builds replayed from a graph that is updated for new lists, other charges and
another precision equal the eager builds, with eager work and host
synchronisations in between, on one stream or several, without waiting for
earlier builds; contexts that work at the same time do not share
work arrays."""
import ctypes as C

import numpy as np
import pytest

from fireball_hip import synth
from fireball_hip.lib import HS_MATS, Assembler
from test_zz_no_alloc import DeviceArrays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("charged", [False, True])
def test_updated_graph_equals_eager_builds(charged):
    sp = synth.CHNO_SPECIES
    st = synth.random_box(synth.chno_counts(40), 1.0, 0.9, 5, sp)
    other = st.ratom + np.random.default_rng(2).normal(0.0, 0.02, st.ratom.shape)
    dq = np.random.default_rng(3).normal(0.0, 0.05, (2, st.natoms, 4)) * np.array([1.0, 1.0, 0.0, 0.0])

    def build(asm, k):
        if charged:
            q = np.ascontiguousarray(dq[k % 2])
            asm._check(asm.L.fb_set_charges(asm.h, 0, q.ctypes.data_as(C.POINTER(C.c_double))))
        asm.assemble_all()
        return {m: asm.blocks(m) for m in HS_MATS}

    asm = Assembler(synth.make_tables(sp), precision="fp64")
    asm.add_structure(st)
    for step in range(3):
        asm.set_positions(0, other if step % 2 else st.ratom)
        asm.build_lists()
        for precision in ("fp64", "mixed"):
            asm.set_precision(precision)
            asm.enable_timing(True)   # eager launches
            eager = [build(asm, k) for k in range(2)]
            asm.timings(64)
            asm.enable_timing(False)
            for k in range(4):
                got = build(asm, k)
                for m in HS_MATS:
                    assert np.array_equal(got[m], eager[k % 2][m]), (step, precision, k, m)
                if k == 1:
                    asm.assemble_S()
                    asm.synchronize()
    asm.close()


class Hip:
    """Streams (default priority) and events of the HIP runtime."""
    NOT_READY = 600

    def __init__(self):
        self.lib = C.CDLL("libamdhip64.so")

    def call(self, name, *args):
        assert getattr(self.lib, name)(*args) == 0, name

    def stream(self):
        s = C.c_void_p()
        self.call("hipStreamCreateWithFlags", C.byref(s), C.c_uint(1))
        return s

    def event(self):
        e = C.c_void_p()
        self.call("hipEventCreateWithFlags", C.byref(e), C.c_uint(2))
        return e


def silicon(stream):
    """1728 atoms on a stream, and the blocks of both precisions."""
    asm = Assembler(synth.make_tables([synth.SI]), precision="mixed")
    asm._check(asm.L.fb_set_stream(asm.h, stream))
    asm.add_structure(synth.diamond_si((6, 6, 6), sigma=0.05, seed=2))
    asm.build_lists()
    want = {}
    for p in ("mixed", "fp64"):
        asm.set_precision(p)
        asm.assemble_all()
        want[p] = {m: asm.blocks(m) for m in HS_MATS}
    return asm, want


def test_a_change_of_precision_does_not_wait_for_earlier_builds():
    hip = Hip()
    stream, ev = hip.stream(), hip.event()
    asm, want = silicon(stream)
    for _ in range(100):   # some 20 ms of binary64 builds
        asm.assemble_all(sync=False)
    hip.call("hipEventRecord", ev, stream)
    asm.set_precision("mixed")
    asm.assemble_all(sync=False)
    state = hip.lib.hipEventQuery(ev)
    asm.synchronize()
    for m in HS_MATS:
        assert np.array_equal(asm.blocks(m), want["mixed"][m]), m
    asm.close()
    assert state == Hip.NOT_READY


def test_builds_on_two_streams_in_turn():
    """Each stream waits on the device for the other's last build; the host waits for none."""
    hip = Hip()
    streams, ev = [hip.stream(), hip.stream()], hip.event()
    asm, want = silicon(streams[0])
    for turn in range(3):
        for k in range(8):
            p = ("mixed", "fp64")[(k // 2 + turn) % 2]
            asm.set_precision(p)
            for _ in range(3):
                asm.assemble_all(sync=False)
            hip.call("hipEventRecord", ev, streams[k % 2])
            hip.call("hipStreamWaitEvent", streams[1 - k % 2], ev, C.c_uint(0))
            asm._check(asm.L.fb_set_stream(asm.h, streams[1 - k % 2]))
        asm.synchronize()
        for m in HS_MATS:
            assert np.array_equal(asm.blocks(m), want[p][m]), (turn, m)
    asm.assemble_all(sync=False)
    asm._check(asm.L.fb_set_stream(asm.h, streams[1]))
    asm.close()   # waits for the stream that was left


def test_charges_are_not_sent_into_a_capture():
    """The call is refused, the capture goes on, and the next build has the charges."""
    hip = Hip()
    stream = hip.stream()
    sp = synth.CHNO_SPECIES
    st = synth.random_box(synth.chno_counts(40), 1.0, 0.9, 5, sp)
    synth.random_dQ([st], sp)
    asm = Assembler(synth.make_tables(sp), precision="fp64")
    asm._check(asm.L.fb_set_stream(asm.h, stream))
    asm.add_structure(st)
    asm.build_lists()
    asm.set_tuning(2, 0)   # direct launches: a build can be captured by the caller
    vna = []

    def charges(scale):
        q = np.ascontiguousarray(scale * st.dQ)
        asm._check(asm.L.fb_set_charges(asm.h, 0, q.ctypes.data_as(C.POINTER(C.c_double))))

    for scale in (1.0, 2.0, 3.0):
        charges(scale)
        asm.assemble_all()
        vna.append(asm.blocks("VNA"))
    for scale, call in ((1.0, asm.L.fb_assemble_all), (2.0, asm.L.fb_assemble_vna_2c)):
        charges(scale)
        hip.call("hipStreamBeginCapture", stream, C.c_int(1))
        graph = C.c_void_p()
        try:
            assert call(asm.h) == -9   # FB_E_HIP
        finally:
            hip.call("hipStreamEndCapture", stream, C.byref(graph))
            hip.call("hipGraphDestroy", graph)
        for again in (scale, 3.0):
            charges(again)
            asm.assemble_all()
            assert np.array_equal(asm.blocks("VNA"), vna[int(again) - 1])
    # with the charges sent, a captured build is the build
    hip.call("hipStreamBeginCapture", stream, C.c_int(1))
    graph = C.c_void_p()
    try:
        asm.assemble_all(sync=False)
    finally:
        hip.call("hipStreamEndCapture", stream, C.byref(graph))
    hip.call("hipGraphDestroy", graph)
    asm.close()


def test_gradients_of_many_contexts_do_not_share_work_arrays():
    """Seven contexts, each on its own stream, more than the library's fixed
    scratch has parts: enqueued together, each with its own parameters, targets,
    batch and element count.  Gradients and losses are those of serial calls."""
    rng = np.random.default_rng(4)
    nm, ts = 8576, synth.make_tables([synth.SI])
    rows, nme = [2048, 1999, 1024, 2048, 700, 1500, 2033], [10, 3, 10, 1, 10, 3, 10]
    asms = [Assembler(ts, precision="mixed") for _ in range(7)]
    with DeviceArrays() as d:
        P = [d.put(0.2 * rng.standard_normal(nm)) for _ in asms]
        X = d.put(rng.uniform(-1.0, 1.0, (2048, 3)))
        T = [d.put(rng.normal(0.0, 0.5, (n, 64))) for n in rows]
        G, loss = [d.filled(nm, 0.0) for _ in asms], [d.filled(1, 0.0) for _ in asms]

        def gradients(together):
            for k, a in enumerate(asms):
                a.mlp_gradients_noalloc(nme[k], P[k], rows[k], X, T[k], G[k], loss[k])
                if not together:
                    a.synchronize()
            for a in asms:
                a.synchronize()
            return [(d.get(g, nm), d.get(x, 1)) for g, x in zip(G, loss)]

        want = gradients(False)
        assert len({float(w[1][0]) for w in want}) == len(want)
        for _ in range(20):
            for got, w in zip(gradients(True), want):
                assert np.array_equal(got[0], w[0]) and np.array_equal(got[1], w[1])
        for a in asms:
            a.close()


def test_captured_gradients_outlive_their_context():
    """Captured in the first and in the sixth context of seven (a fixed and a
    further part of the scratch), replayed after all are destroyed, with eager
    work and synchronisations between the replays."""
    hip = Hip()
    rng = np.random.default_rng(8)
    n, nm, ts = 700, 8576, synth.make_tables([synth.SI])
    with DeviceArrays() as d:
        X, T = d.put(rng.uniform(-1.0, 1.0, (n, 3))), d.put(rng.normal(0.0, 0.5, (n, 64)))
        P = [d.put(0.2 * rng.standard_normal(nm)) for _ in range(2)]
        G, loss = [d.filled(nm, 0.0) for _ in P], [d.filled(1, 0.0) for _ in P]
        asms = [Assembler(ts, precision="mixed") for _ in range(7)]
        stream, execs, want = hip.stream(), [], []
        for k, a in enumerate((asms[0], asms[5])):
            a.mlp_gradients_noalloc(10, P[k], n, X, T, G[k], loss[k])
            a.synchronize()
            want.append((d.get(G[k], nm), d.get(loss[k], 1)))
            a._check(a.L.fb_set_stream(a.h, stream))
            g, e = C.c_void_p(), C.c_void_p()
            hip.call("hipStreamBeginCapture", stream, C.c_int(1))
            a.mlp_gradients_noalloc(10, P[k], n, X, T, G[k], loss[k])
            hip.call("hipStreamEndCapture", stream, C.byref(g))
            hip.call("hipGraphInstantiate", C.byref(e), g, None, None, C.c_size_t(0))
            execs.append(e)
        for a in asms:
            a.close()
        other = Assembler(ts, precision="mixed")   # has one of the parts
        other.add_structure(synth.diamond_si((2, 2, 2), sigma=0.05, seed=2))
        for _ in range(4):
            zero = np.zeros(nm, np.float32)
            for k in range(2):
                hip.call("hipMemcpy", C.c_void_p(G[k]), zero.ctypes.data_as(C.c_void_p), C.c_size_t(zero.nbytes),
                         C.c_int(1))
                hip.call("hipGraphLaunch", execs[k], stream)
            hip.call("hipStreamSynchronize", stream)
            for k in range(2):
                assert np.array_equal(d.get(G[k], nm), want[k][0])
                assert np.array_equal(d.get(loss[k], 1), want[k][1])
            other.build_lists()
            other.assemble_all()
            other.mlp_gradients_noalloc(10, P[0], n, X, T, G[1], loss[1])
            other.synchronize()
            assert np.array_equal(d.get(G[1], nm), want[0][0])
        for e in execs:
            hip.call("hipGraphExecDestroy", e)
        other.close()
