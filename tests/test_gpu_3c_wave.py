"""The binary64 three-centre kernels at the edges of their tiles: segments
shorter than, equal to and longer than the 64 triplets of a pass, lists of
mixed pair classes, third atoms with one and two shells, shells without
charge.  The blocks equal the oracle's, bit for bit."""
import numpy as np
import pytest

import oracle
from fireball_hip import synth
from fireball_hip.lib import HS_MATS, Assembler

pytestmark = pytest.mark.gpu


def droplet(n, species, radius=2.8, seed=11, rmin=0.65):
    rng = np.random.default_rng(seed)
    pos = []
    while len(pos) < n:
        p = rng.uniform(-radius, radius, 3)
        if p @ p < radius * radius and all(np.linalg.norm(p - q) > rmin for q in pos):
            pos.append(p)
    imass = rng.integers(1, len(species) + 1, n).astype(np.int32)
    return synth.Structure(np.array(pos) + 20.0, imass, np.diag([40.0] * 3), 1)


@pytest.mark.parametrize("n", [3, 17, 65, 66, 67, 69])
@pytest.mark.parametrize("charged", [False, True])
def test_bcna_bits(n, charged):
    sp = synth.CHNO_SPECIES if n < 60 else [synth.SI, synth.H_SP]
    st = droplet(n, sp)
    if charged:
        synth.random_dQ([st], sp)
        st.dQ[::3] = 0.0        # atoms without charge, and shells without
        st.dQ[1::3, 0] = 0.0
    ts = synth.make_tables(sp)
    asm = Assembler(ts, precision="fp64")
    asm.add_structure(st)
    asm.build_lists()
    asm.assemble_all()
    o = oracle.System(oracle.Tables(ts), st).run_all()
    for m in HS_MATS:
        assert np.array_equal(asm.blocks(m), o[m]), m


@pytest.mark.parametrize("n", [3, 17, 66])
def test_bcna_bits_of_shell_charges_that_cancel(n):
    st = droplet(n, [synth.SI])
    st.dQ = np.zeros((n, 4))
    st.dQ[:, 0] = np.random.default_rng(5).uniform(0.1, 0.4, n)
    st.dQ[:, 1] = -st.dQ[:, 0]
    st.dQ[3::4] = 0.0
    ts = synth.make_tables([synth.SI])
    asm = Assembler(ts, precision="fp64")
    asm.add_structure(st)
    asm.build_lists()
    asm.assemble_all()
    o = oracle.System(oracle.Tables(ts), st).run_all()
    for m in HS_MATS:
        assert np.array_equal(asm.blocks(m), o[m]), m


@pytest.mark.parametrize("n", [3, 17, 66, 67])
def test_density_bits(n):
    sp = synth.CHNO_SPECIES if n < 60 else [synth.SI, synth.H_SP]
    st = droplet(n, sp)
    ts = synth.add_rho_tables(synth.make_tables(sp))
    qin = synth.shell_qin(st, sp)
    asm = Assembler(ts, precision="fp64")
    asm.add_structure(st)
    asm.build_lists()
    asm.set_qin(qin)
    asm.assemble_rho(("ALL",))
    s = oracle.System(oracle.Tables(ts), st)
    s.build_lists()
    o = s.run_rho(qin)
    for m in ("RHO_IN", "RHO_BOND", "RHOW_IN", "RHOW_BOND"):
        assert np.array_equal(asm.rho(m), o[m]), m
