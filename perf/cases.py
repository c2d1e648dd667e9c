"""The work a user has this framework do, as cases that can be timed and checked.

A case is a dict of plain values: a `kind` (which entry points a pass calls), a
`system` with its sizes, and the options of the call.  The kinds:

  build    one H+S build (S, T, dipole_z, Vna 2c and 3c) on lists that exist;
           with charges, new shell charges are set first, as one iteration of
           a self-consistent loop does
  step     one geometry step: new positions, neighbour and triplet lists, H+S
  forces   density matrix in, force build, force pieces (and Dblocks) out
  rho      new shell charges in, McWEDA density build, four block arrays out
  pp       one geometry step of the pseudopotential: lists, sVNL, vnl, blocks out
  mlp      one forward and backward pass of the learned 3c surrogate

Systems: diamond Si supercells (one species, s and p shells), random C/H/N/O
boxes (four species, s and sp, every pair class), amorphous carbon, and a
batch of structures of both families.  The seed draws the tables, the shell
charges, the density matrix and where the structure lies (a translation and a
symmetry of the cube); the geometry up to that symmetry belongs to the case,
so that the lists of every seed have the same lengths.

H+S blocks come back as the library's device arrays.  Where the interface
hands results to the host, they go to page-locked arrays that the state keeps,
as a program that calls the interface in a loop keeps them.
"""
from __future__ import annotations

import ctypes as C
import functools
import itertools
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "thunder-master_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from fireball_hip import synth  # noqa: E402
from fireball_hip.lib import FB_MAT, HS_MATS, Assembler, lib  # noqa: E402

P_EQ2 = synth.P_EQ2
RHO_MATS = ("RHO_IN", "RHO_BOND", "RHOW_IN", "RHOW_BOND")
MLP_SIZES = (64 * 3, 64, 64 * 64, 64, 64 * 64, 64)   # W1, b1, W2, b2, W3, b3
MLP_NP = sum(MLP_SIZES)


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # the smallest periodic cell in use: launch and call costs count
        {"name": "build_si64", "kind": "build", "system": "si", "n1": 2, "n2": 2, "n3": 2, "precision": "mixed",
         "charged": False},
        # the headline workload: 4096 atoms, mixed precision, neutral
        {"name": "build_si4096", "kind": "build", "system": "si", "n1": 8, "n2": 8, "n3": 8, "precision": "mixed",
         "charged": False},
        # a large organic box in binary64: every pair class, the reference's arithmetic
        {"name": "build_chno3000_fp64", "kind": "build", "system": "chno", "natoms": 3000, "precision": "fp64",
         "charged": False},
        # one self-consistency iteration of an ordinary charged system, odd size
        {"name": "scf_chno501", "kind": "build", "system": "chno", "natoms": 501, "precision": "mixed",
         "charged": True},
        # many independent structures of 16 to 1024 atoms as one batch
        {"name": "build_batch48", "kind": "build", "system": "batch", "nstruct": 48, "precision": "mixed",
         "charged": False},
        # a molecular-dynamics step of a small box: lists of a small system
        {"name": "step_chno96", "kind": "step", "system": "chno", "natoms": 96, "precision": "mixed"},
        # a step of dense amorphous carbon: 62 neighbours per atom, 3.4 million triplets
        {"name": "step_c2048", "kind": "step", "system": "carbon", "natoms": 2048, "precision": "mixed"},
        # Vna forces of a crystal, mixed 3c interpolation
        {"name": "forces_si1728", "kind": "forces", "system": "si", "n1": 6, "n2": 6, "n3": 6, "precision": "mixed",
         "charged": False, "dblocks": False},
        # forces and every Dblock of a charged droplet (no periodic images), binary64
        {"name": "forces_drop151_fp64", "kind": "forces", "system": "drop", "natoms": 151, "precision": "fp64",
         "charged": True, "dblocks": True},
        # McWEDA densities of a crystal, binary64 as the entry points always are
        {"name": "rho_si1728", "kind": "rho", "system": "si", "n1": 6, "n2": 6, "n3": 6},
        # pseudopotential of an organic box: lists and blocks of a new geometry
        {"name": "pp_chno1000", "kind": "pp", "system": "chno", "natoms": 1000},
        # one training step's gradients of the surrogate, the largest batch of the entry point
        {"name": "mlp_grad2048", "kind": "mlp", "batch": 2048, "nme": 10},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_si(rng, most):
    while True:
        n = [rng.randint(2, 8) for _ in range(3)]
        if 8 * n[0] * n[1] * n[2] <= most:
            return {"system": "si", "n1": n[0], "n2": n[1], "n3": n[2]}


def _draw_box(rng, most, drop=False):
    if not drop and rng.random() < 0.4:
        return _draw_si(rng, most)
    return {"system": "drop" if drop else "chno", "natoms": _log_int(rng, 40, most)}


def draw(rng):
    kind = rng.choice(("build", "build", "batch", "step", "forces", "rho", "pp", "mlp"))
    prec = rng.choice(("mixed", "mixed", "fp64"))
    if kind == "batch":
        return {"kind": "build", "system": "batch", "nstruct": _log_int(rng, 4, 48), "precision": prec,
                "charged": False}
    if kind == "mlp":
        return {"kind": "mlp", "batch": _log_int(rng, 16, 2048), "nme": rng.choice((1, 3, 10))}
    if kind == "build":
        charged = rng.random() < 0.4
        return dict(_draw_box(rng, 1000 if charged else 3000), kind="build", precision=prec, charged=charged)
    if kind == "step":
        if rng.random() < 0.25:
            return {"kind": "step", "system": "carbon", "natoms": _log_int(rng, 200, 2048), "precision": prec}
        return dict(_draw_box(rng, 3000), kind="step", precision=prec)
    if kind == "forces":
        small = rng.random() < 0.4
        return dict(_draw_box(rng, 200 if small else 1500, drop=small), kind="forces", precision=prec,
                    charged=rng.random() < 0.4, dblocks=small)
    return dict(_draw_box(rng, 1500 if kind == "rho" else 1000), kind=kind)


# ------------------------------------------------------------------ the inputs
@functools.lru_cache(maxsize=64)
def _geometry(key):
    """The structures of a case, before the seed's translation and symmetry."""
    case = dict(key)
    if case["system"] == "si":
        return [synth.diamond_si((case["n1"], case["n2"], case["n3"]), sigma=0.08, seed=17)]
    if case["system"] == "carbon":
        return [synth.random_box({6: case["natoms"]}, 2.0, 1.2, 3, [synth.C_SP])]
    if case["system"] == "batch":
        return synth.batch_structures(case["nstruct"], seed=2)
    s = synth.random_box(synth.chno_counts(case["natoms"]), 1.0, 0.9, 1, synth.CHNO_SPECIES)
    s.icluster = 1 if case["system"] == "drop" else 0
    return [s]


def _species(case):
    sp = {"si": [synth.SI], "carbon": [synth.C_SP], "batch": synth.batch_species()}.get(case["system"],
                                                                                      synth.CHNO_SPECIES)
    return synth.with_pp(sp) if case["kind"] == "pp" else sp


def _base(case):
    return _geometry(tuple(sorted((k, v) for k, v in case.items() if k in ("system", "n1", "n2", "n3", "natoms",
                                                                        "nstruct"))))


def _placed(st, rng):
    """The structure under a random axis permutation, reflections and translation."""
    perm, sign = rng.permutation(3), rng.choice((-1.0, 1.0), 3)
    box = np.diag(st.lattice)[perm]
    ratom = st.ratom[:, perm] * sign + rng.uniform(0.0, 1.0, 3) * box
    return synth.Structure(np.ascontiguousarray(ratom), st.imass.copy(), np.diag(box), st.icluster, name=st.name)


def _shell_values(st, species, rng, neutral):
    """Shell charges [natoms][4]: deviations within 0.05 e, on top of the neutral occupations for Qin."""
    occ = np.zeros((len(species), 4))
    has = np.zeros((len(species), 4))
    for i, sp in enumerate(species):
        has[i, :sp.nssh] = 1.0
        if neutral:
            occ[i, :sp.nssh] = synth.QNEUTRAL[sp.nZ][:sp.nssh]
    k = st.imass - 1
    return occ[k] + has[k] * rng.uniform(-0.05, 0.05, (st.natoms, 4))


def _inputs(case, seed):
    """Everything a pass computes from, on the host: the same for prepare() and exact()."""
    rng = np.random.default_rng([seed, 9])
    if case["kind"] == "mlp":
        lim = [1 / math.sqrt(3)] * 2 + [1 / 8] * 4
        params = np.concatenate([rng.uniform(-b, b, n) for n, b in zip(MLP_SIZES, lim)])
        X = rng.uniform(-1.0, 1.0, (case["batch"], 3))
        T = rng.uniform(-1.0, 1.0, (case["batch"], 64))
        return [a.astype(np.float32) for a in (params, X, T)]
    species = _species(case)
    ts = synth.make_tables(species, seed=int(rng.integers(1 << 30)))
    if case["kind"] == "rho":
        synth.add_rho_tables(ts, seed=int(rng.integers(1 << 30)))
    if case["kind"] == "pp":
        synth.add_pp_tables(ts, seed=int(rng.integers(1 << 30)))
    structs = [_placed(s, rng) for s in _base(case)]
    charges = None
    if case.get("charged") or case["kind"] == "rho":
        charges = [_shell_values(s, species, rng, case["kind"] == "rho") for s in structs]
    return ts, structs, charges, rng


def _density(rng, blen):
    return rng.uniform(-0.5, 0.5, blen)


# ------------------------------------------------------------------ the program
class _DeviceArray:
    """A device array of the library as torch takes it, without a copy; torch keeps this object, and with it
    the context that owns the memory, for as long as a tensor uses it."""

    def __init__(self, asm, ptr, n):
        self.asm = asm
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": "<f8", "data": (ptr, False), "version": 3}


def _device_blocks(state):
    """The five H+S block arrays of the context; the views are made again when the library moved them."""
    asm, views = state["asm"], state["views"]
    ptr, n = C.c_void_p(), C.c_int64()
    out = {}
    for m in HS_MATS:
        asm._check(asm.L.fb_get_device_blocks(asm.h, FB_MAT[m], C.byref(ptr), C.byref(n)))
        key = (ptr.value, n.value)
        if views.get(m, (None,))[0] != key:
            views[m] = (key, torch.as_tensor(_DeviceArray(asm, *key), device="cuda"))
        out[m] = views[m][1]
    return out


def _pinned(n, like=None):
    t = torch.empty(max(int(n), 1), dtype=torch.float64, pin_memory=True)
    if like is not None:
        t.copy_(torch.from_numpy(like))
    return t


def _dp(t):
    return C.cast(t.data_ptr(), C.POINTER(C.c_double))


def _len(asm, fn, istruct=0):
    n = C.c_int64()
    asm._check(fn(asm.h, istruct, C.byref(n)))
    return n.value


def prepare(case, seed):
    if case["kind"] == "mlp":
        species = [synth.SI]
        asm = Assembler(synth.make_tables(species), precision="mixed")
        p, X, T = (torch.from_numpy(a).cuda() for a in _inputs(case, seed))
        return {"kind": "mlp", "asm": asm, "n": case["batch"], "nme": case["nme"], "p": p, "X": X, "T": T,
                "grads": torch.zeros(MLP_NP, device="cuda"), "loss": torch.zeros(1, device="cuda")}
    ts, structs, charges, rng = _inputs(case, seed)
    kind = case["kind"]
    asm = Assembler(ts, precision=case.get("precision", "fp64"))
    state = {"kind": kind, "asm": asm, "views": {}, "charges": charges, "dblocks": case.get("dblocks")}
    moves = kind in ("step", "pp")
    for s in structs:
        dq = charges[len(asm.structs)] if charges and kind != "rho" else None
        # where the program moves the atoms, the lists that it has are those of the step before
        before = s.ratom + np.random.default_rng([seed, 4]).normal(0.0, 0.01, s.ratom.shape) if moves else s.ratom
        asm.add_structure(synth.Structure(before, s.imass, s.lattice, s.icluster, dQ=dq))
    asm.build_lists()
    if kind in ("build", "step", "forces"):
        asm.assemble_all()
    if moves:
        state["ratom"] = structs[0].ratom
    L = asm.L
    if kind == "forces":
        blen = _len(asm, L.fb_get_block_len)
        npairs, n = asm.list_sizes()[0], structs[0].natoms
        state["rho"] = _pinned(blen, _density(rng, blen))
        state["out"] = {k: _pinned(3 * m) for k, m in (("vna_atom", npairs), ("vna_ontop", npairs), ("f3naa", n),
                                                     ("f3nab", n), ("f3nac", n))}
        if case["dblocks"]:
            state["out"].update({"D" + m: _pinned(3 * blen) for m in ("S", "T", "DIP")})
    if kind == "rho":
        asm.set_qin(charges[0])
        b, w = _len(asm, L.fb_get_block_len), _len(asm, L.fb_get_shell_block_len)
        state["out"] = {m: _pinned(w if m.startswith("RHOW") else b) for m in RHO_MATS}
    if kind == "pp":
        asm.build_lists_pp()
        sz = asm.pp_sizes()
        state["out"] = {"SVNL": _pinned(sz[4] + 4096), "VNL": _pinned(sz[5] + 4096)}
    return state


def run(state):
    kind, asm = state["kind"], state["asm"]
    L, h = asm.L, asm.h
    if kind == "mlp":
        asm.mlp_gradients_noalloc(state["nme"], state["p"].data_ptr(), state["n"], state["X"].data_ptr(),
                                  state["T"].data_ptr(), state["grads"].data_ptr(), state["loss"].data_ptr())
        return state["grads"], state["loss"]
    if kind == "build":
        if state["charges"]:
            for k, q in enumerate(state["charges"]):
                asm._check(L.fb_set_charges(h, k, q.ctypes.data_as(C.POINTER(C.c_double))))
        asm.assemble_all(sync=False)
        return _device_blocks(state)
    if kind == "step":
        asm.set_positions(0, state["ratom"])
        asm.build_lists()
        asm.assemble_all(sync=False)
        return _device_blocks(state)
    out = state["out"]
    if kind == "forces":
        asm._check(L.fb_set_denmat(h, 0, _dp(state["rho"])))
        asm.dassemble_all()
        asm._check(L.fb_get_forces(h, 0, *(_dp(out[k]) for k in ("vna_atom", "vna_ontop", "f3naa", "f3nab", "f3nac"))))
        if state["dblocks"]:
            for m in ("S", "T", "DIP"):
                asm._check(L.fb_get_dblocks(h, 0, FB_MAT[m], _dp(out["D" + m])))
        return out
    if kind == "rho":
        asm.set_qin(state["charges"][0])
        asm.assemble_rho(("ALL",))
        for m in RHO_MATS:
            asm._check(L.fb_get_blocks(h, 0, FB_MAT[m], _dp(out[m])))
        return out
    asm.set_positions(0, state["ratom"])
    asm.build_lists()
    asm.build_lists_pp()
    asm.assemble_pp()
    sz = asm.pp_sizes()
    for k, m in enumerate(("SVNL", "VNL")):
        if sz[4 + k] > out[m].numel():
            out[m] = _pinned(sz[4 + k])
        asm._check(L.fb_get_pp_blocks(h, 0, k, _dp(out[m])))
    return {m: out[m][:sz[4 + k]] for k, m in enumerate(("SVNL", "VNL"))}


# ------------------------------------------------------------------ what a pass cannot do without
def _counts(case):
    """Atoms, pairs, triplets and block elements of a case, from its densities: neighbours lie in a sphere
    of the cutoff, triplets are ordered pairs of neighbours within the cutoff of each other."""
    tot = np.zeros(4)
    species = _species(case)
    rc = np.array([max(sp.rcutoffA) for sp in species])
    norb = np.array([sp.norb for sp in species], float)
    for s in _base(case):
        k = s.imass - 1
        r = 2.0 * rc[k].mean() - 0.01
        vol = abs(np.linalg.det(s.lattice))
        if s.icluster == 1:
            r = min(r, 0.62 * vol ** (1.0 / 3.0))
        nn = s.natoms / vol * 4.0 / 3.0 * math.pi * r ** 3
        # 15/32: the mean overlap of the cutoff spheres of two atoms within one cutoff
        tot += (s.natoms, s.natoms * (nn + 1.0), s.natoms * nn * nn * 15.0 / 32.0,
                s.natoms * (nn + 1.0) * norb[k].mean() ** 2)
    return tot


def work(case):
    """Inputs read once and outputs written once; operations of the interpolations and rotations alone."""
    kind = case["kind"]
    if kind == "mlp":
        n = case["batch"]
        return {"bytes": 4.0 * (n * (3 + 64) + 2 * MLP_NP + 1), "flops": 2.0 * n * (3 * (64 * 3 + 2 * 64 * 64) - 64 * 3)}
    atoms, pairs, trips, blen = _counts(case)
    shells = 3.0 if case.get("charged") else 1.0
    two = 700.0 * pairs * (3.0 + 3.0 * shells)      # 7 points x 10 elements and a rotation per interaction
    three = 900.0 * trips * shells                  # 5 theta x 3 points x 10 elements and a rotation
    if kind in ("build", "step"):
        lists = 16.0 * pairs + 20.0 * trips
        return {"bytes": 56.0 * atoms + lists + 40.0 * blen, "flops": two + three}
    if kind == "forces":
        return {"bytes": 24.0 * atoms + 8.0 * blen * (10.0 if case["dblocks"] else 1.0) + 64.0 * pairs + 20.0 * trips
                + 72.0 * atoms, "flops": 4.0 * two + 8.0 * three}
    if kind == "rho":
        return {"bytes": 56.0 * atoms + 16.0 * pairs + 20.0 * trips + 20.0 * blen, "flops": 2.0 * two + 3.0 * three}
    pp = 0.45 * blen       # projector cutoffs are shorter than orbital ones; vnl reaches further
    return {"bytes": 24.0 * atoms + 8.0 * (pp + 2.6 * blen), "flops": 700.0 * pairs + 130.0 * 1.4 * trips}


def tolerance(case):
    """About four times what the path shows against 64 bits over the ranges of draw()."""
    if case["kind"] == "mlp":
        return {"rel": 5e-7}                      # FP32 sums over up to 2048 samples: 1.1e-7
    if case["kind"] == "forces":                  # binary64 2e-12 (derivatives of the frames), mixed 7e-8
        return {"rel": 6e-7, "max": 6e-5} if case["precision"] == "mixed" else {"rel": 1e-11, "max": 1e-9}
    if case.get("precision") == "mixed":          # FP32 interpolation of the 3c term: 3e-9 of the Vna blocks
        return {"rel": 4e-8, "max": 4e-6}
    return {"rel": 1e-13, "max": 1e-11}           # binary64 sums in another order: 1e-14


# ------------------------------------------------------------------ the same in plain torch, 64 bits
def _sum_at(out, index, values):
    out.index_add_(0, index.reshape(-1), values.reshape(-1))


class _Plain:
    """The assembly of one structure in plain binary64 torch, by its definitions."""

    CHUNK = 100000

    def __init__(self, ts, st, charges=None):
        self.dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
        self.ts, self.st, self.sp = ts, st, ts.species
        t = functools.partial(torch.as_tensor, device=self.dev)
        self.r = t(st.ratom, dtype=torch.float64)
        self.im = t(st.imass.astype(np.int64)) - 1
        self.lat = t(st.lattice, dtype=torch.float64)
        self.rc = t([max(s.rcutoffA) for s in self.sp], dtype=torch.float64)
        self.rcmin = t([min(s.rcutoffA) for s in self.sp], dtype=torch.float64)
        self.norb = t([s.norb for s in self.sp])
        self.q = None if charges is None else t(charges, dtype=torch.float64)
        # images as integer triples, image 0 at the origin, then x fastest
        box = [(0, 0, 0)]
        if st.icluster != 1:
            box += [(x, y, z) for z, y, x in itertools.product(range(-4, 5), repeat=3) if (x, y, z) != (0, 0, 0)]
        self.img = t(box)
        self.xl = self.img.to(torch.float64) @ self.lat
        self.img_id = torch.full((9, 9, 9), -1, dtype=torch.int64, device=self.dev)
        self.img_id[self.img[:, 0] + 4, self.img[:, 1] + 4, self.img[:, 2] + 4] = torch.arange(len(box), device=self.dev)
        self.pi, self.pb, self.pj = self.neighbours(self.rc, self.rc)
        self.pdisp = self.r[self.pj] + self.xl[self.pb] - self.r[self.pi]
        self.pself = (self.pi == self.pj) & (self.pb == 0)
        self.boff, self.blen = self.offsets(self.norb[self.im[self.pi]] * self.norb[self.im[self.pj]])
        self.self_of = torch.empty(len(self.r), dtype=torch.int64, device=self.dev)
        self.self_of[self.pi[self.pself]] = torch.nonzero(self.pself)[:, 0]
        self.tables = {}

    @staticmethod
    def offsets(sizes):
        end = torch.cumsum(sizes, 0)
        return end - sizes, int(end[-1])

    def neighbours(self, rci, rcj):
        """(atom, image, neighbour) with |r_j + xl - r_i| < rci + rcj - 0.01, in that order."""
        ri, rj = rci[self.im], rcj[self.im]
        lo, hi = self.r.min(0).values, self.r.max(0).values
        reach = (float(ri.max()) + float(rj.max()))
        found = []
        for b in range(len(self.xl)):
            gap = torch.maximum(lo + self.xl[b] - hi, lo - (hi + self.xl[b])).clamp(min=0)
            if float(gap.norm()) > reach:
                continue
            for i0 in range(0, len(self.r), 2048):
                d = self.r[None] + self.xl[b] - self.r[i0:i0 + 2048, None]
                near = d.square().sum(-1).sqrt() < ri[i0:i0 + 2048, None] + rj[None] - 0.01
                i, j = torch.nonzero(near, as_tuple=True)
                found.append(torch.stack((i + i0, torch.full_like(i, b), j)))
        got = torch.cat(found, 1)
        return got[:, torch.argsort((got[0] * len(self.xl) + got[1]) * len(self.r) + got[2])]

    def image(self, triple):
        """Image number of an integer triple, -1 outside the image set."""
        inside = (triple.abs() <= 4).all(-1)
        c = triple.clamp(-4, 4) + 4
        return torch.where(inside, self.img_id[c[:, 0], c[:, 1], c[:, 2]], torch.full_like(c[:, 0], -1))

    def pair_index(self, pairs, i, b, j):
        """Position of (i, b, j) in a list of neighbours() and whether it is there."""
        n = len(self.r)
        keys = (pairs[0] * len(self.xl) + pairs[1]) * n + pairs[2]
        want = (i * len(self.xl) + b) * n + j
        at = torch.searchsorted(keys, want).clamp(max=len(keys) - 1)
        return at, (b >= 0) & (keys[at] == want)

    @staticmethod
    def ordered_pairs(owner, n):
        """All (p, q) of list entries with the same owner; owner is sorted."""
        cnt = torch.bincount(owner, minlength=n)
        start = torch.cumsum(cnt, 0) - cnt
        p = torch.repeat_interleave(torch.arange(len(owner), device=owner.device), cnt[owner])
        first = torch.cumsum(cnt[owner], 0) - cnt[owner]
        q = start[owner[p]] + torch.arange(len(p), device=owner.device) - first[p]
        return p, q

    def triplets(self):
        """(third atom, pair-list entries of the two others, target pair) of every common-neighbour triplet."""
        p, q = self.ordered_pairs(self.pi, len(self.r))
        ok = (p != q) & ~self.pself[p] & ~self.pself[q]
        p, q = p[ok], q[ok]
        ia, ja = self.pj[p], self.pj[q]
        d = (self.pdisp[q] - self.pdisp[p]).square().sum(-1).sqrt()
        ok = d < self.rc[self.im[ia]] + self.rc[self.im[ja]] - 0.01
        p, q = p[ok], q[ok]
        b = self.image(self.img[self.pb[q]] - self.img[self.pb[p]])
        tgt, ok = self.pair_index((self.pi, self.pb, self.pj), self.pj[p], b, self.pj[q])
        return self.pi[p[ok]], p[ok], q[ok], tgt[ok]

    # -- interpolation
    def table2(self, key):
        if key not in self.tables:
            c = self.ts.cells2c[key]
            self.tables[key] = (c, torch.as_tensor(c.data, device=self.dev))
        return self.tables[key]

    def elements2(self, key, z, shape):
        """Molecular-frame block [n, mu, nu] of a two-centre table: 7-point Lagrange."""
        c, data = self.table2(key)
        dx = c.xmax / (c.nx - 1)
        left = ((z.detach() / dx).long() - 3).clamp(0, c.nx - 7)
        node = left[:, None] + torch.arange(7, device=self.dev)
        u = z[:, None] - node.to(z.dtype) * dx
        F = 0.0
        for i in range(7):
            L = torch.ones_like(z)
            for j in range(7):
                if j != i:
                    L = L * u[:, j] / ((i - j) * dx)
            F = F + L[:, None] * data[node[:, i]]
        return self.to_block(c, F, shape)

    def to_block(self, c, F, shape):
        at = torch.as_tensor((c.mu - 1) * shape[1] + (c.nu - 1), device=self.dev).long()
        M = torch.zeros(len(F), shape[0] * shape[1], dtype=torch.float64, device=self.dev)
        return M.index_copy(1, at, F).view(-1, *shape)

    def table3(self, key):
        if key not in self.tables:
            cells = [self.ts.cells3c[key + (th,)] for th in range(1, 6)]
            data = np.stack([c.data for c in cells], 2)            # [iy, ix, theta, ME]
            self.tables[key] = (cells[0], torch.as_tensor(data, device=self.dev))
        return self.tables[key]

    def elements3(self, key, x, y, cost, shape):
        """Molecular-frame block of a three-centre table: bicubic, or the plane through three points where
        the gradient of the first element is below 1e-6; the plane's slopes are those of that first element."""
        c, data = self.table3(key)
        dx, dy = c.xmax / (c.nx - 1.0), c.ymax / (c.ny - 1.0)
        ix = ((x.detach() / dx).long() + 1).clamp(2, c.nx - 2) - 1
        iy = ((y.detach() / dy).long() + 1).clamp(2, c.ny - 2) - 1
        px, py = x / dx - ix, y / dy - iy
        gx = (data[iy, ix + 1, 0, 0] - data[iy, ix, 0, 0]) / dx
        gy = (data[iy + 1, ix, 0, 0] - data[iy, ix, 0, 0]) / dy
        plane = gx * gx + gy * gy < 1e-6

        def cubic(p):
            return ((p - 0) * (p - 1) * (p - 2) / -6, (p + 1) * (p - 1) * (p - 2) / 2, (p + 1) * p * (p - 2) / -2,
                    (p + 1) * p * (p - 1) / 6)

        wx, wy = cubic(px), cubic(py)
        flat = {(0, 0): (1 - px - py).detach(), (1, 0): px.detach(), (0, 1): py.detach()}
        F = 0.0
        for i, j in itertools.product(range(4), repeat=2):
            w = torch.where(plane, flat.get((i - 1, j - 1), torch.zeros_like(px)), wx[i] * wy[j])
            F = F + w[:, None, None] * data[iy + j - 1, ix + i - 1]
        slope = torch.where(plane, gx * (x - x.detach()) + gy * (y - y.detach()), torch.zeros_like(x))
        F = F + slope[:, None, None]
        c2 = cost * cost
        P = torch.stack((torch.ones_like(cost), cost, 0.5 * (3 * c2 - 1), 0.5 * cost * (5 * c2 - 3),
                         0.125 * (3 - c2 * (30 - 35 * c2))), 1)
        F = (P[:, :, None] * F).sum(1)
        s0 = (1 - c2.detach()).clamp(min=1e-5).sqrt()
        sint = s0 - cost.detach() / s0 * (cost - cost.detach())
        odd = torch.as_tensor(c.mvalue == 1, device=self.dev)
        return self.to_block(c, torch.where(odd, F * sint[:, None], F), shape)

    # -- frames and rotations (orbitals s, then p as y, z, x)
    @staticmethod
    def rotation(yp, zp):
        xp = torch.linalg.cross(yp, zp)
        axes = torch.stack((yp, zp, xp), 2)[:, [1, 2, 0]]
        R = torch.zeros(len(zp), 4, 4, dtype=zp.dtype, device=zp.device)
        R[:, 0, 0] = 1.0
        R[:, 1:, 1:] = axes
        return R

    @classmethod
    def bond_rotation(cls, d, z, side=None):
        """z' along the bond; y' = z' x side.  The tables do not depend on the sign of m, so that any side gives
        the same block; those of the projectors do, and the side is then the second atom's position."""
        up = torch.zeros_like(d)
        up[:, 2] = 1.0
        zp = torch.where(z[:, None] < 1e-5, up, d / z.clamp(min=1e-12)[:, None])
        if side is None:
            side = torch.nn.functional.one_hot(zp.detach().abs().argmin(1), 3).to(d.dtype)
        yp = torch.linalg.cross(zp, side)
        return cls.rotation(yp / yp.norm(dim=1, keepdim=True), zp)

    @staticmethod
    def rotate(R, M):
        return R[:, :M.shape[1], :M.shape[1]] @ M @ R[:, :M.shape[2], :M.shape[2]].transpose(1, 2)

    def groups(self, *species):
        """Indices of the entries of every species combination that occurs."""
        key = functools.reduce(lambda a, b: a * len(self.sp) + b, species)
        for k in torch.unique(key).tolist():
            which = []
            for _ in species:
                which.insert(0, k % len(self.sp))
                k //= len(self.sp)
            at = torch.nonzero(key == functools.reduce(lambda a, b: a * len(self.sp) + b, which))[:, 0]
            for part in torch.split(at, self.CHUNK):
                yield part, [self.sp[w] for w in which], [w + 1 for w in which]

    @staticmethod
    def smoother(r, rend):
        ratio = (r - 0.8 * rend) / (0.2 * rend)
        s = (1 - ratio * ratio) ** 2
        return torch.where(r > rend, torch.zeros_like(r), torch.where(r < 0.8 * rend, torch.ones_like(r), s))

    @staticmethod
    def put(off, X):
        """Places and values of blocks in the flat column-major layout."""
        v = X.transpose(1, 2).reshape(len(X), -1)
        return off[:, None] + torch.arange(v.shape[1], device=v.device), v

    def pair_groups(self, keep):
        idx = torch.nonzero(keep)[:, 0]
        for part, sp, ids in self.groups(self.im[self.pi[idx]], self.im[self.pj[idx]]):
            yield idx[part], sp, ids

    def trip_groups(self):
        al, p, q, tgt = self.triplets()
        for part, sp, ids in self.groups(self.im[self.pj[p]], self.im[self.pj[q]], self.im[al]):
            yield al[part], p[part], q[part], tgt[part], sp, ids

    def shell_sum(self, term, nssh, charge):
        """Neutral term (subtype 0) plus the charged subtypes."""
        X = term(0)
        if self.q is not None:
            for s in range(nssh):
                X = X + charge[:, s, None, None] * term(s + 1, True)
        return X

    # -- H+S
    def simple(self, itype, ids, d, z, shape):
        return self.rotate(self.bond_rotation(d, z), self.elements2((*ids, itype, 0), z, shape))

    def ontop(self, ids, sp, d, z, i, j):
        R, shape = self.bond_rotation(d, z), (sp[0].norb, sp[1].norb)
        q = self.q if self.q is not None else torch.zeros(len(self.r), 4, device=self.dev)
        X = 0.0
        for itype, s, at in ((synth.P_VNA_ONTOPL, sp[0], i), (synth.P_VNA_ONTOPR, sp[1], j)):
            X = X + self.shell_sum(lambda k, _=False: self.elements2((*ids, itype, k), z, shape), s.nssh, q[at])
        return self.rotate(R, X) * P_EQ2

    def atom_term(self, ids, sp, d, z, j, sself):
        R, shape = self.bond_rotation(d, z), (sp[0].norb, sp[0].norb)
        smooth = self.smoother(z, float(self.rcmin[ids[0] - 1] + self.rcmin[ids[1] - 1]))[:, None, None]
        far = sself / z.clamp(min=1e-4)[:, None, None] * (z > 1e-4)[:, None, None]

        def term(k, charged=False):
            X = self.rotate(R, self.elements2((*ids, synth.P_VNA_ATOM, k), z, shape))
            return (1 - smooth) * far + smooth * X if charged else X

        q = self.q if self.q is not None else torch.zeros(len(self.r), 4, device=self.dev)
        return self.shell_sum(term, sp[1].nssh, q[j]) * P_EQ2

    def bcna(self, ids, sp, ra, r1, r2, q):
        """Three-centre block of the positions of the third atom and the two others."""
        shape = (sp[0].norb, sp[1].norb)
        d, c = r2 - r1, ra - (r1 + r2) / 2
        z, x = d.norm(dim=1), c.norm(dim=1)
        zp, rh = d / z[:, None], c / x[:, None]
        cost = (zp * rh).sum(1)
        yp = torch.linalg.cross(zp, rh)
        yp = yp / yp.norm(dim=1, keepdim=True)
        R = self.rotation(yp, zp)
        guard = torch.linalg.cross(d, c).norm(dim=1) < 1e-3     # frames count as constant on a line
        R = torch.where(guard[:, None, None], R.detach(), R)
        if self.q is not None:
            d13, d23 = (ra - r1).norm(dim=1), (ra - r2).norm(dim=1)
            rend = [float(self.rcmin[ids[k] - 1] + self.rcmin[ids[2] - 1]) for k in (0, 1)]
            stinky = (self.smoother(d13, rend[0]) * self.smoother(d23, rend[1]))[:, None, None]
            S = self.simple(synth.P_OVERLAP, ids[:2], d, z, shape) / 2
            D = self.simple(synth.P_DIPOLE_Z, ids[:2], d, z, shape) / z[:, None, None]
            far = (S - D) / d13[:, None, None] + (S + D) / d23[:, None, None]

        def term(k, charged=False):
            X = self.rotate(R, self.elements3((*ids, synth.P_BCNA, k), x, z, cost, shape))
            return stinky * X + (1 - stinky) * far if charged else X

        return self.shell_sum(term, sp[2].nssh, q) * P_EQ2

    def trip_points(self, al, p, q):
        ra = self.r[al]
        return ra, ra + self.pdisp[p], ra + self.pdisp[q]

    def charge_of(self, at):
        return None if self.q is None else self.q[at]

    def zeros(self, n):
        return torch.zeros(n, dtype=torch.float64, device=self.dev)

    def hs(self):
        out = {m: self.zeros(self.blen) for m in HS_MATS}
        every = torch.ones_like(self.pself)
        for at, sp, ids in self.pair_groups(every):
            d, shape = self.pdisp[at], (sp[0].norb, sp[1].norb)
            z = d.norm(dim=1)
            for m, it in (("S", synth.P_OVERLAP), ("T", synth.P_KINETIC), ("DIP", synth.P_DIPOLE_Z)):
                _sum_at(out[m], *self.put(self.boff[at], self.simple(it, ids, d, z, shape)))
            other = at[~self.pself[at]]
            if len(other):
                d2 = self.pdisp[other]
                X = self.ontop(ids, sp, d2, d2.norm(dim=1), self.pi[other], self.pj[other])
                _sum_at(out["VNAO"], *self.put(self.boff[other], X))
        for at, sp, ids in self.pair_groups(every):
            d = self.pdisp[at]
            own = self.boff[self.self_of[self.pi[at]]]
            X = self.atom_term(ids, sp, d, d.norm(dim=1), self.pj[at], self.self_blocks(out["S"], own, sp[0].norb))
            _sum_at(out["VNA"], *self.put(own, X))
        for al, p, q, tgt, sp, ids in self.trip_groups():
            X = self.bcna(ids, sp, *self.trip_points(al, p, q), self.charge_of(al))
            _sum_at(out["VNA"], *self.put(self.boff[tgt], X))
        return out

    @staticmethod
    def self_blocks(S, off, n):
        return S[off[:, None] + torch.arange(n * n, device=S.device)].view(-1, n, n).transpose(1, 2)

    # -- forces: minus the gradient of density times block, by autograd
    def density_blocks(self, rho, off, shape):
        at = off[:, None] + torch.arange(shape[0] * shape[1], device=self.dev)
        return rho[at].view(-1, shape[1], shape[0]).transpose(1, 2)

    def forces(self, rho, dblocks):
        rho = torch.as_tensor(rho, device=self.dev)
        n, npairs = len(self.r), len(self.pi)
        out = {k: self.zeros((m, 3)) for k, m in (("vna_atom", npairs), ("vna_ontop", npairs), ("f3naa", n),
                                                ("f3nab", n), ("f3nac", n))}
        if dblocks:
            out.update({"D" + m: self.zeros(3 * self.blen) for m in ("S", "T", "DIP")})
        S = self.zeros(self.blen)
        for at, sp, ids in self.pair_groups(self.pself):
            d = self.pdisp[at]
            _sum_at(S, *self.put(self.boff[at], self.simple(synth.P_OVERLAP, ids, d, d.norm(dim=1),
                                                            (sp[0].norb, sp[1].norb))))
        for at, sp, ids in self.pair_groups(~self.pself):
            shape = (sp[0].norb, sp[1].norb)
            own = self.boff[self.self_of[self.pi[at]]]
            r1 = torch.zeros_like(self.pdisp[at]).requires_grad_()
            d = self.pdisp[at] - r1
            z = d.norm(dim=1)
            E = (self.density_blocks(rho, self.boff[at], shape) *
                 self.ontop(ids, sp, d, z, self.pi[at], self.pj[at])).sum()
            out["vna_ontop"][at] = -torch.autograd.grad(E, r1, retain_graph=True)[0]
            E = (self.density_blocks(rho, own, (shape[0], shape[0])) *
                 self.atom_term(ids, sp, d, z, self.pj[at], self.self_blocks(S, own, shape[0]))).sum()
            out["vna_atom"][at] = -torch.autograd.grad(E, r1, retain_graph=True)[0]
            if dblocks:
                for m, it in (("S", synth.P_OVERLAP), ("T", synth.P_KINETIC), ("DIP", synth.P_DIPOLE_Z)):
                    X = self.simple(it, ids, d, z, shape)
                    for mu, nu in itertools.product(range(shape[0]), range(shape[1])):
                        g = torch.autograd.grad(X[:, mu, nu].sum(), r1, retain_graph=True)[0]
                        first = 3 * (self.boff[at] + nu * shape[0] + mu)
                        out["D" + m][first[:, None] + torch.arange(3, device=self.dev)] = g
        for al, p, q, tgt, sp, ids in self.trip_groups():
            ra, r1, r2 = (r.detach() for r in self.trip_points(al, p, q))
            ra.requires_grad_()
            r1.requires_grad_()
            V = self.bcna(ids, sp, ra, r1, r2, self.charge_of(al))
            E = (self.density_blocks(rho, self.boff[tgt], (sp[0].norb, sp[1].norb)) * V).sum()
            ga, gb = torch.autograd.grad(E, (ra, r1))
            out["f3naa"].index_add_(0, al, -ga)
            out["f3nab"].index_add_(0, self.pj[p], -gb)
            out["f3nac"].index_add_(0, self.pj[q], ga + gb)
        return {k: v.reshape(-1) for k, v in out.items()}

    # -- McWEDA densities: Qin-weighted sums over the shells of the contributing atom
    def densities(self):
        out = {}
        nssh = torch.as_tensor([s.nssh for s in self.sp], device=self.dev)
        woff, wlen = self.offsets(nssh[self.im[self.pi]] * nssh[self.im[self.pj]])
        for pre, types, off, total in (("RHO", (15, 16, 17, 1), self.boff, self.blen),
                                       ("RHOW", (19, 20, 21, 2), woff, wlen)):
            whole = pre == "RHO"
            rin, bond = self.zeros(total), self.zeros(total)
            size = (lambda s: s.norb) if whole else (lambda s: s.nssh)

            def term(M, R):
                return self.rotate(R, M) if whole else M

            for at, sp, ids in self.pair_groups(torch.ones_like(self.pself)):
                d = self.pdisp[at]
                z = d.norm(dim=1)
                R = self.bond_rotation(d, z)
                X = 0.0
                for itype, s, who in ((types[0], sp[0], self.pi), (types[1], sp[1], self.pj)):
                    for k in range(s.nssh):
                        M = self.elements2((*ids, itype, k + 1), z, (size(sp[0]), size(sp[1])))
                        X = X + self.q[who[at], k][:, None, None] * term(M, R)
                X = X * (~self.pself[at])[:, None, None]
                for o in (rin, bond):
                    _sum_at(o, *self.put(off[at], X))
                X = 0.0
                for k in range(sp[1].nssh):
                    M = self.elements2((*ids, types[2], k + 1), z, (size(sp[0]), size(sp[0])))
                    X = X + self.q[self.pj[at], k][:, None, None] * term(M, R)
                own = off[self.self_of[self.pi[at]]]
                _sum_at(rin, *self.put(own, X))
                _sum_at(bond, *self.put(own, X * self.pself[at][:, None, None]))
            for al, p, q, tgt, sp, ids in self.trip_groups():
                ra, r1, r2 = self.trip_points(al, p, q)
                d, c = r2 - r1, ra - (r1 + r2) / 2
                z, x = d.norm(dim=1), c.norm(dim=1)
                zp, rh = d / z[:, None], c / x[:, None]
                yp = torch.linalg.cross(zp, rh)
                R = self.rotation(yp / yp.norm(dim=1, keepdim=True), zp)
                X = 0.0
                for k in range(sp[2].nssh):
                    M = self.elements3((*ids, types[3], k + 1), x, z, (zp * rh).sum(1), (size(sp[0]), size(sp[1])))
                    X = X + self.q[al, k][:, None, None] * term(M, R)
                _sum_at(rin, *self.put(off[tgt], X))
            out[pre + "_IN"], out[pre + "_BOND"] = rin, bond
        return out

    # -- pseudopotential: vnl = sum over projector atoms of P cl P^T
    def pseudo(self):
        rpp = torch.as_tensor([s.rcutoff_pp for s in self.sp], dtype=torch.float64, device=self.dev)
        npp = torch.as_tensor([s.norb_pp for s in self.sp], device=self.dev)
        cl = self.zeros((len(self.sp), 4))
        for i, s in enumerate(self.sp):
            row = [c for c, l in zip(s.cl_pp, s.lssh_pp) for _ in range(2 * l + 1)]
            cl[i, :len(row)] = torch.as_tensor(row, dtype=torch.float64)
        pp, px = self.neighbours(self.rc, rpp), self.neighbours(rpp, self.rc)
        soff, slen = self.offsets(self.norb[self.im[pp[0]]] * npp[self.im[pp[2]]])
        svnl = self.zeros(slen)
        P = self.zeros((pp.shape[1], 4, 4))              # orbital, projector; zero beyond a species' own
        d = self.r[pp[2]] + self.xl[pp[1]] - self.r[pp[0]]
        for at, sp, ids in self.groups(self.im[pp[0]], self.im[pp[2]]):
            shape = (sp[0].norb, sp[1].norb_pp)
            z = d[at].norm(dim=1)
            R = self.bond_rotation(d[at], z, self.r[pp[0][at]] + d[at])
            X = self.rotate(R, self.elements2((*ids, synth.P_VNL, 0), z, shape))
            _sum_at(svnl, *self.put(soff[at], X))
            P[at, :shape[0], :shape[1]] = X
        # every (atom, projector atom, atom): through the projector atom's own PPx list, in list order
        cnt = torch.bincount(px[0], minlength=len(self.r))
        start = torch.cumsum(cnt, 0) - cnt
        per = cnt[pp[2]]
        a = torch.repeat_interleave(torch.arange(pp.shape[1], device=self.dev), per)
        b = start[pp[2][a]] + torch.arange(len(a), device=self.dev) - (torch.cumsum(per, 0) - per)[a]
        i, j = pp[0][a], px[2][b]
        image = self.image(self.img[pp[1][a]] + self.img[px[1][b]])
        key = (i * len(self.xl) + image) * len(self.r) + j
        uniq, inv = torch.unique(key, return_inverse=True)
        seen = torch.full((len(uniq),), len(a), dtype=torch.int64, device=self.dev)
        seen.scatter_reduce_(0, inv, torch.arange(len(a), device=self.dev), "amin")
        order = torch.argsort(seen)
        first = seen[order]
        voff, vlen = self.offsets(self.norb[self.im[i[first]]] * self.norb[self.im[j[first]]])
        place = torch.empty_like(order)
        place[order] = torch.arange(len(order), device=self.dev)
        back, _ = self.pair_index(pp, j, self.image(-self.img[px[1][b]]), pp[2][a])
        vnl = self.zeros(vlen)
        for at, sp, _ in self.groups(self.im[i], self.im[j]):
            X = (P[a[at]] * cl[self.im[pp[2][a[at]]]][:, None, :]) @ P[back[at]].transpose(1, 2)
            _sum_at(vnl, *self.put(voff[place[inv[at]]], X[:, :sp[0].norb, :sp[1].norb]))
        return {"SVNL": svnl, "VNL": vnl}


def _exact_mlp(case, seed):
    p, X, T = (torch.as_tensor(a.astype(np.float64)) for a in _inputs(case, seed))
    p.requires_grad_()
    W1, b1, W2, b2, W3, b3 = torch.split(p, MLP_SIZES)

    def act(z):
        c = z.clamp(-4.0, 4.0)
        return z * (0.5 + c * (0.25 - c.abs() / 32.0))

    a = act(X @ W1.view(64, 3).T + b1)
    a = act(a @ W2.view(64, 64).T + b2)
    Y = a @ W3.view(64, 64).T + b3
    # output slot o holds theta r % 5 of matrix element (o >> 2 & 3) + 4 (r // 5), r = 4 (o >> 4) + (o & 3)
    valid = []
    for o in range(64):
        r = 4 * (o >> 4) + (o & 3)
        valid.append(r // 5 < 3 and ((o >> 2) & 3) + 4 * (r // 5) < case["nme"])
    valid = torch.tensor(valid)
    loss = (Y - T)[:, valid].square().mean()
    loss.backward()
    return p.grad, loss.detach().reshape(1)


def exact(case, seed):
    kind = case["kind"]
    if kind == "mlp":
        return _exact_mlp(case, seed)
    ts, structs, charges, rng = _inputs(case, seed)
    if kind in ("build", "step"):
        parts = [_Plain(ts, s, charges[k] if charges else None).hs() for k, s in enumerate(structs)]
        return {m: torch.cat([p[m] for p in parts]) for m in HS_MATS}
    plain = _Plain(ts, structs[0], charges[0] if charges else None)
    if kind == "forces":
        return plain.forces(_density(rng, plain.blen), case["dblocks"])
    return plain.densities() if kind == "rho" else plain.pseudo()
