"""Neighbour and triplet lists where their kernels can go wrong: neighbour
counts either side of a wavefront and of a workgroup, cells of one atom,
ragged batches, lattices whose images coincide.  Lists and binary64 blocks
equal the oracle's."""
import numpy as np
import pytest

import oracle
from fireball_hip import synth
from fireball_hip.lib import HS_MATS, Assembler

pytestmark = pytest.mark.gpu

LISTS = ("neighn", "neigh_j", "neigh_b", "neigh_back", "neigh_self", "ncommon", "com_iatom_j", "com_iatom_b",
         "com_jatom_j", "com_jatom_b", "com_mneigh")


def check(species, structs):
    ts = synth.make_tables(species)
    asm = Assembler(ts, precision="fp64")
    for st in structs:
        asm.add_structure(st)
    asm.build_lists()
    asm.assemble_all()
    tables = oracle.Tables(ts)
    for k, st in enumerate(structs):
        o = oracle.System(tables, st).run_all()
        r = asm.run_all(k)
        for name in LISTS:
            assert np.array_equal(r[name], o[name]), (k, name)
        for m in HS_MATS:
            assert np.array_equal(r[m], o[m]), (k, m)
    asm.close()


def droplet(n, species, radius, seed=3, rmin=0.7):
    """n atoms of random species in a ball, no two closer than rmin."""
    rng = np.random.default_rng(seed)
    pos = []
    while len(pos) < n:
        p = rng.uniform(-radius, radius, 3)
        if p @ p < radius * radius and all(np.linalg.norm(p - q) > rmin for q in pos):
            pos.append(p)
    imass = rng.integers(1, len(species) + 1, n).astype(np.int32)
    return synth.Structure(np.array(pos) + 20.0, imass, np.diag([40.0] * 3), 1)


@pytest.mark.parametrize("n", [1, 2, 3, 62, 63, 64, 65, 66])
def test_neighbours_around_a_wavefront(n):
    """Every atom sees every other: lists of n entries, segments of n - 2 triplets."""
    check([synth.SI], [droplet(n, [synth.SI], 2.8)])


def test_ragged_batch_of_periodic_and_cluster_structures():
    sp = synth.CHNO_SPECIES
    box = synth.random_box(synth.chno_counts(37), 1.0, 0.9, 5, sp)
    wide = synth.Structure(box.ratom.copy(), box.imass.copy(), np.diag([9.0, 30.0, 60.0]), 0)
    skew = synth.Structure(box.ratom.copy(), box.imass.copy(),
                           np.array([[11.0, 0.0, 0.0], [3.0, 10.0, 0.0], [-2.0, 4.0, 12.0]]), 0)
    one = synth.Structure(np.array([[1.0, 2.0, 3.0]]), np.array([2], np.int32), np.diag([3.1, 4.2, 5.3]), 0)
    check(sp, [box, droplet(70, sp, 4.5), one, wide, skew])


def test_lattice_with_coincident_images():
    """6 a1 + 5 a2 = 0: different image numbers name one point, the lists are still those of the reference's scan."""
    lat = np.array([[12.0, 0.0, 0.0], [-14.4, 0.0, 0.0], [0.0, 0.0, 12.0]])
    pos = np.array([[1.0, 0.3, 0.2], [1.0, 0.1, 0.9], [1.0, 1.4, 0.5]])   # apart across the repeat of 2.4 A only
    check([synth.H_SP], [synth.Structure(pos, np.ones(3, np.int32), lat, 0)])


@pytest.mark.parametrize("n", [255, 256, 257])
def test_neighbours_around_the_capacity_of_the_one_pass_search(n):
    """Every atom sees every other, so the lists are known."""
    g = 0.62 * np.array(np.meshgrid(*[np.arange(-5, 6)] * 3)).reshape(3, -1).T
    pos = g[np.argsort(np.sum(g * g, axis=1), kind="stable")[:n]]
    pos += np.random.default_rng(1).uniform(-0.03, 0.03, pos.shape)
    asm = Assembler(synth.make_tables([synth.SI]), precision="fp64")
    asm.add_structure(synth.Structure(pos + 20.0, np.ones(n, np.int32), np.diag([40.0] * 3), 1))
    asm.build_lists()
    r = asm.lists()
    assert np.all(r["neighn"] == n) and np.all(r["neigh_b"] == 0)
    assert np.array_equal(r["neigh_j"].reshape(n, n), np.tile(np.arange(1, n + 1), (n, 1)))
    assert np.array_equal(r["neigh_back"].reshape(n, n), np.tile(np.arange(1, n + 1)[:, None], (1, n)))
    assert np.array_equal(r["neigh_self"], np.arange(1, n + 1))
    asm.close()


def test_more_atoms_than_one_workgroup_bins():
    spatial = pytest.importorskip("scipy.spatial")
    st = synth.diamond_si((11, 11, 11), sigma=0.05, seed=4)
    asm = Assembler(synth.make_tables([synth.SI]), precision="fp64")
    asm.add_structure(st)
    asm.build_lists()
    r = asm.lists()
    box = np.diag(st.lattice)
    x = np.mod(st.ratom, box)
    tree = spatial.cKDTree(x, boxsize=box)
    rng = 2.0 * max(synth.SI.rcutoffA) - 0.01
    count = np.array([len(q) for q in tree.query_ball_point(x, rng)])
    assert np.array_equal(r["neighn"], count)
    # neigh_back is an involution between the pairs
    off = np.concatenate([[0], np.cumsum(r["neighn"])])
    back = off[r["neigh_j"] - 1] + r["neigh_back"] - 1
    assert np.array_equal(back[back], np.arange(len(back)))
    asm.close()
