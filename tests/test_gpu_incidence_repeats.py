"""Lists that name an atom more than once in a row, through both paths of the list-built incidence.

Each repeated slot is an edge of its own (the pack keeps every one), so the plain scheme's fold has
to pair slots one to one whichever path builds the lists: hash tables in LDS, or a sort of the bin's
entries (rows past 1,760 slots, bins that more entries name than LDS holds, rows that repeat an atom
whose own row names them back). Rows repeat some of their neighbours once or twice, some in both
directions and some in one; in the longer cases a third of the rows is filled with atoms past the
cutoff, many of them repeated too, up to the length under test, and `hubs` gives every row far atoms
of the first bin, whose entries then fit LDS no more. Against the oracle, and rebuilds of the
same list bit for bit."""

from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from lk_testutil import assert_energy, assert_forces, assert_virial
from lammps_jax_amd import harness, systems
from lammps_jax_amd.pair import PairJax

pytestmark = pytest.mark.gpu


def _far(x, xi, cutoff):
    return np.flatnonzero(np.sum((x - xi) ** 2, axis=1) > (cutoff + 0.1) ** 2)


def _repeating(sysm, cutoff, longest, hubs):
    """The system's list with repeated entries (and far ones, see above)."""
    rng = np.random.default_rng(17)
    lst = dict(sysm.list)
    stride, room = lst["stride"], lst["maxneighs"]
    old = np.asarray(lst["neighbors"]).reshape(room, stride) & 0x3FFFFFFF
    num = np.array(lst["numneigh"], copy=True)
    x = sysm.x[:sysm.nall]
    rows = {int(i): old[:num[i], i].tolist() for i in np.asarray(lst["ilist"])[:lst["inum"]]}
    owned = list(rows)
    for i in rng.choice(owned, len(owned) // 2, replace=False).tolist():
        j = int(rng.choice(old[:num[i], i]))
        for _ in range(int(rng.integers(1, 3))):
            rows[i].insert(int(rng.integers(0, len(rows[i]) + 1)), j)
        if j in rows and i in rows[j] and rng.random() < 0.5:
            rows[j].insert(int(rng.integers(0, len(rows[j]) + 1)), i)
    for n, i in enumerate(owned):
        rows[i] += _far(x[:hubs], x[i], cutoff).tolist()
        if n % 3 == 0 and len(rows[i]) < longest:
            rows[i] = np.resize(_far(x, x[i], cutoff), longest - len(rows[i])).tolist() + rows[i]
    room = max(len(r) for r in rows.values())
    nb = np.zeros((room, stride), np.int32)
    for i, r in rows.items():
        nb[:len(r), i] = r
        num[i] = len(r)
    lst.update(neighbors=np.ascontiguousarray(nb.reshape(-1)), numneigh=num, maxneighs=room)
    sysm.list = lst
    return lst


CASES = [  # scheme, precision, cells, longest row, hubs
    ("plain", 8, (4, 4, 4), 0, 0),
    ("plain", 4, (7, 5, 4), 0, 0),
    ("plain", 8, (5, 4, 4), 1800, 0),
    ("plain", 4, (9, 8, 8), 0, 12),
    ("plain", 8, (18, 18, 18), 0, 12),  # 270,000 entries of one bin: its marks leave LDS too
    ("half", 8, (4, 5, 4), 0, 0),
    ("half", 4, (4, 4, 4), 2050, 0),
    ("half", 8, (9, 8, 8), 0, 12),
]


def _check(sysm, wl_cutoff, lst, model, scheme, precision, max_atoms=None):
    half = scheme == "half"
    pj = PairJax(sysm, model, precision=precision, accumulation=scheme, max_atoms=max_atoms,
                 max_edges=128 * sysm.nall)
    print(f"repeated entries {scheme} precision={precision} room={lst['maxneighs']} "
          f"nall={sysm.nall} capacity={pj.max_atoms}", flush=True)
    pos, sp = O.pack_atoms(sysm.x, sysm.type, sysm.nall, sysm.nall, precision)
    s, r, m, count, _ = O.pack_neighbors(sysm.x, lst, max_atoms=sysm.nall,
                                         max_edges=pj.max_edges, nlocal=sysm.nlocal,
                                         cutoff=wl_cutoff)
    kw = dict(nlocal=sysm.nlocal, nghost=sysm.nghost, senders=s, receivers=r, mask=m,
              precision=precision)
    if half:
        ref = O.eam_compute(model[1], pos, sp, ghost_owner=sysm.ghost_owner, mode=O.HALF, **kw)
    else:
        ref = O.lj_compute(model[1], pos, mode=O.PLAIN, **kw)
    nall = sysm.nall
    first = None
    for fused in (True, True, True, False):
        info = pj.compute(fused=fused)
        f = pj.forces().copy()
        assert info.edge_count == count
        assert_energy(precision, info.energy, ref["energy"], sysm.nlocal)
        assert_forces(precision, f[:nall], ref["forces"][:nall])
        assert_virial(precision, info.virial, O.virial_fdotr(ref["forces"][:nall], sysm.x, nall))
        if first is None:
            first = (info.energy, f)
        assert info.energy == first[0] and np.array_equal(f, first[1])
        pj.list_epoch += 1  # the engine's rebuild signal: the same lists again
        pj.h.set_list_epoch(pj.list_epoch)


@pytest.mark.parametrize("scheme,precision,cells,longest,hubs", CASES)
def test_repeated_entries(gpu, scheme, precision, cells, longest, hubs):
    half = scheme == "half"
    wl = systems.make_workload("eam_alloy_8k" if half else "lj_ghost_262k", cells=cells, seed=21)
    sysm = systems.System(wl.x, wl.types, wl.box, wl.cutoff + wl.skin)
    sysm.build_list(wl.cutoff + wl.skin, kind=harness.LIST_HALF if half else harness.LIST_FULL)
    lst = _repeating(sysm, wl.cutoff, longest, hubs)
    _check(sysm, wl.cutoff, lst, ("eam", wl.tables) if half else ("lj", wl.lj), scheme, precision)


@pytest.mark.parametrize("scheme,precision", [("plain", 4), ("plain", 8), ("half", 8)])
def test_capacity_past_32_bit_entries(gpu, scheme, precision):
    """A contract of more than 2^26 - 1 atoms, whose entries travel in 64 bits; rows of at most 32
    slots, which is what such a capacity leaves of the validity bits' 27-bit addresses."""
    half = scheme == "half"
    a = 3.8 if half else 1.68
    cutoff, skin = (3.5, 0.5) if half else (1.6, 0.2)
    box = np.full(3, 6 * a)
    rng = np.random.default_rng(2)
    x = systems.fcc_lattice(6, 6, 6, a)
    x = systems.wrap(x + rng.normal(0.0, 0.03 * a, size=x.shape), box)
    types = rng.integers(1, 3, len(x)).astype(np.int32) if half else np.ones(len(x), np.int32)
    sysm = systems.System(x, types, box, cutoff + skin)
    sysm.build_list(cutoff + skin, kind=harness.LIST_HALF if half else harness.LIST_FULL)
    lst = _repeating(sysm, cutoff, 0, 0)
    assert lst["maxneighs"] <= 32, lst["maxneighs"]
    model = (("eam", systems.synthetic_alloy_tables(cutoff=cutoff)) if half else
             ("lj", dict(epsilon=1.0, sigma=1.0, cutoff=cutoff, edge_energy_scale=0.5)))
    _check(sysm, cutoff, lst, model, scheme, precision, max_atoms=(1 << 26) + 1000)
