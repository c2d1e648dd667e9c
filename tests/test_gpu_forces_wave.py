"""The s/p three-centre force kernels where their work is split: tiles shorter
than, equal to and longer than the 64 triplets of a pass, lists of mixed pair
classes, third atoms and shells without charge, more neighbours than one pass
of the per-atom sums holds, and near-collinear triplets on both sides of the
limits of epsilon's fallback frame and of Depsilon_3c.

The oracle contracts derivative blocks, the kernels take the gradient of one
number per triplet; both are binary64 sums of some hundred terms per triplet
and of up to 1e4 triplets per atom, so they agree to a few 1e-13 of the largest
term: 1e-11 of the largest per-atom force, as for the golden cases.  Added to
it is the oracle's own rounding (Depsilon_3c divides z^2 a - (a.d) d, which
cancels, by crossmag^2): for the most collinear triplet 2^-53 z^2 |a| /
crossmag^2 of its rotational energy, eight products of rho and V of at most 1,
times the 14.4 of the forces' unit.  Against an evaluation in 80-bit arithmetic the oracle is
8.5e-11 off for 65 atoms and the kernels 1.4e-13."""
import numpy as np
import pytest

import oracle
from fireball_hip import synth
from fireball_hip.lib import Assembler

pytestmark = pytest.mark.gpu


def oracle_rounding(st):
    """2^-53 z^2 |a| / crossmag^2 of the most collinear triplet with a rotational part, times 8 * 14.4"""
    r, worst = st.ratom, 0.0
    for i in range(len(r)):
        d, a = r - r[i], r - r[i]
        z = np.linalg.norm(d, axis=1)
        cm = np.linalg.norm(np.cross(d[:, None], a[None]), axis=2)
        ok = cm >= 1e-3
        q = np.where(ok, (z * z)[:, None] * z[None] / np.where(ok, cm, 1.0) ** 2, 0.0)
        worst = max(worst, q.max())
    return 2.0 ** -53 * worst * 8 * 14.4


def compare(ts, st, most=0, precision="fp64", rel=1e-11, roundings=1):
    s = oracle.System(oracle.Tables(ts), st)
    lists = s.run_all()
    assert max(lists["neighn"]) > most
    rho = synth.denmat(ts.species, st.imass, lists["neighn"], lists["neigh_j"], lists["neigh_back"])
    ref = s.run_forces(rho)
    asm = Assembler(ts, precision=precision)
    asm.add_structure(st)
    asm.build_lists()
    asm.assemble_all()
    asm.set_denmat(rho)
    asm.dassemble_all()
    f = asm.forces()
    extra = roundings * oracle_rounding(st)
    for k in ("f3naa", "f3nab", "f3nac"):
        tol = rel * max(1.0, float(np.max(np.abs(ref[k])))) + extra
        np.testing.assert_allclose(f[k], ref[k], rtol=0, atol=tol, err_msg=k)
    return ref


def droplet(n, species, radius=2.8, rmin=0.65):
    rng = np.random.default_rng(11)
    pos = []
    while len(pos) < n:
        p = rng.uniform(-radius, radius, 3)
        if p @ p < radius * radius and all(np.linalg.norm(p - q) > rmin for q in pos):
            pos.append(p)
    imass = rng.integers(1, len(species) + 1, n).astype(np.int32)
    return synth.Structure(np.array(pos) + 20.0, imass, np.diag([40.0] * 3), 1)


@pytest.mark.parametrize("n", [3, 17, 65, 66, 67, 69, 140])
@pytest.mark.parametrize("charged", [False, True])
def test_tiles(n, charged):
    sp = synth.CHNO_SPECIES if n < 60 else [synth.SI, synth.H_SP]
    st = droplet(n, sp) if n < 100 else droplet(n, [synth.SI], 2.9, 0.55)
    if charged:
        synth.random_dQ([st], sp)
        st.dQ[::3] = 0.0        # atoms without charge, and shells without
        st.dQ[1::3, 0] = 0.0
    compare(synth.make_tables(sp), st, 128 if n == 140 else 0)


@pytest.mark.parametrize("n", [3, 17, 66])
@pytest.mark.parametrize("precision, rel", [("fp64", 1e-11), ("mixed", 1e-6)])
def test_shell_charges_that_cancel(n, precision, rel):
    """Charge moved from s to p on neutral atoms: no monopole is left, the smoothing's slope times the
    shells' energies is.  Some atoms keep a net charge, some have none.  Mixed precision: a dozen FP32
    roundings (2^-24) of the neutral term, 1e-6 of the largest force.  The oracle's cancelling difference
    carries four roundings of z^2 |a| (of z^2, of a.d, of its product with d and of the difference);
    against 80-bit arithmetic it is 1.1e-11 off for these 17 atoms, 1e-10 for 66."""
    st = droplet(n, [synth.SI])
    st.dQ = np.zeros((n, 4))
    st.dQ[:, 0] = np.random.default_rng(5).uniform(0.1, 0.4, n)
    st.dQ[:, 1] = -st.dQ[:, 0]
    st.dQ[2::4, 1] += 0.1
    st.dQ[3::4] = 0.0
    compare(synth.make_tables([synth.SI]), st, precision=precision, rel=rel, roundings=4)


@pytest.mark.parametrize("sine", [2e-6, 7.4e-5, 8.5e-5, 9.8e-5, 1.02e-4, 1e-3])
@pytest.mark.parametrize("charged", [False, True])
def test_near_collinear(sine, charged):
    # bond of 4.2 A, third atom 1 A behind it: z x = 13 A^2
    sp = [synth.SI]
    axis = np.array([0.48, 0.6, 0.64])
    side = np.cross(axis, [0.0, 0.0, 1.0])
    side /= np.linalg.norm(side)
    pos = np.array([[0.0] * 3, 4.2 * axis, 5.2 * axis + 3.1 * sine * side]) + 20.0
    st = synth.Structure(pos, np.ones(3, np.int32), np.diag([40.0] * 3), 1)
    if charged:
        synth.random_dQ([st], sp)
    ref = compare(synth.make_tables(sp), st)
    assert np.max(np.abs(ref["f3naa"])) > 0.0


@pytest.mark.parametrize("n", [1, 3, 4, 6])
@pytest.mark.parametrize("charged", [False, True])
def test_pair_forces_on_every_route_equal_the_generic_kernels(n, charged):
    """Few, some and many pairs: a workgroup per item, several items per workgroup, a lane per pair."""
    st = synth.diamond_si((n, n, n), sigma=0.05, seed=2)
    if charged:
        synth.random_dQ([st], [synth.SI])
        st.dQ[::5] = 0.0
    ts = synth.make_tables([synth.SI])
    got = []
    for generic in (False, True):
        asm = Assembler(ts, precision="fp64")
        asm.add_structure(st)
        asm.build_lists()
        asm.assemble_all()
        if generic:
            asm.set_tuning(3, 0)
        r = np.random.default_rng(7).normal(0.0, 0.3, len(asm.blocks("S")))
        asm.set_denmat(r)
        asm.dassemble()
        f = asm.forces()
        got.append([asm.dblocks(m) for m in ("S", "T", "DIP")] + [f["vna_atom"], f["vna_ontop"]])
        asm.close()
    for a, b in zip(*got):
        assert np.array_equal(a, b)
