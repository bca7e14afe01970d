"""The pack kernels of the fused steps at the edges of their slots and tiles, against the oracle.

`k_pack_rows` (two-sided and LJ steps) keeps the neighbours of 128 slots of a row in LDS and reads
later ones again, four slots of eight waves at a time; lists with room for more than 256 slots take
`k_step_pack`, whose bits past 256 slots stay in memory. `k_pack_count` and `k_pack_write` (the pack
called on its own) go 256 slots at a time. The rows are cut to, or given far atoms up
to, the lengths under test (the far ones are dropped by the cutoff, so the packed pairs come from
either side of each edge), and the last tile is partly filled. The float32 one-sided EAM step's pack
decides from float records, so a whole neighbour shell is put on its cutoff. Packed pairs bit for
bit after canonical ordering, forces at the usual bars (lk_testutil)."""

from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from lk_testutil import assert_energy, assert_forces, canonical
from lammps_jax_amd import harness, systems
from lammps_jax_amd.pair import PairJax

pytestmark = pytest.mark.gpu


def _resized(sysm, cutoff, longest, width):
    """The system's list with room for `width` slots and every third row given atoms past the
    cutoff, ahead of its own, up to `longest` slots (each third row once more cut to its first)."""
    lst = dict(sysm.list)
    stride, rows = lst["stride"], lst["maxneighs"]
    old = np.asarray(lst["neighbors"]).reshape(rows, stride)
    num = np.array(lst["numneigh"], copy=True)
    room = max(width, rows, longest)
    nb = np.zeros((room, stride), np.int32)
    nb[:rows] = old
    x = sysm.x[:sysm.nall]
    for i in np.asarray(lst["ilist"])[:lst["inum"]:3]:
        far = np.flatnonzero(np.sum((x - x[i]) ** 2, axis=1) > (cutoff + 0.1) ** 2)
        add = max(0, longest - int(num[i]))
        own = old[:num[i], i].copy()
        nb[:add, i] = np.resize(far, add)
        nb[add:add + num[i], i] = own
        num[i] += add
    num[np.asarray(lst["ilist"])[1:lst["inum"]:3]] = 1
    lst.update(neighbors=np.ascontiguousarray(nb.reshape(-1)), numneigh=num, maxneighs=room)
    sysm.list = lst
    return lst


CASES = [  # scheme, precision, cells, longest row, room
    ("plain", 8, (4, 4, 4), 0, 0),
    ("plain", 4, (4, 4, 5), 127, 0),
    ("plain", 8, (4, 4, 4), 128, 0),
    ("plain", 4, (4, 4, 4), 129, 160),
    ("plain", 8, (4, 4, 4), 160, 256),
    ("plain", 4, (5, 4, 4), 256, 256),
    ("plain", 8, (4, 4, 4), 257, 257),
    ("plain", 4, (4, 4, 4), 300, 300),
    ("onesided", 8, (4, 4, 4), 129, 0),
    ("onesided", 4, (5, 5, 4), 256, 0),
    ("onesided", 8, (4, 4, 4), 100, 300),
    ("onesided", 4, (4, 4, 4), 290, 300),
]


@pytest.mark.parametrize("scheme,precision,cells,longest,width", CASES)
def test_pack_rows(gpu, scheme, precision, cells, longest, width):
    wl = systems.make_workload("lj_ghost_262k", cells=cells, seed=9)
    sysm = systems.System(wl.x, wl.types, wl.box, wl.cutoff + wl.skin)
    sysm.build_list(wl.cutoff + wl.skin, kind=harness.LIST_FULL)
    lst = _resized(sysm, wl.cutoff, longest, width)
    pj = PairJax(sysm, ("lj", wl.lj), precision=precision, accumulation=scheme, fused=True)
    print(f"pack rows {scheme} precision={precision} cells={cells} longest={longest} "
          f"room={lst['maxneighs']} nlocal={sysm.nlocal}", flush=True)
    pos, _ = O.pack_atoms(sysm.x, sysm.type, sysm.nall, pj.max_atoms, precision)
    s, r, m, count, _ = O.pack_neighbors(sysm.x, lst, max_atoms=pj.max_atoms,
                                         max_edges=pj.max_edges, nlocal=sysm.nlocal,
                                         cutoff=wl.cutoff)
    ref = O.lj_compute(wl.lj, pos, nlocal=sysm.nlocal, nghost=sysm.nghost, senders=s, receivers=r,
                       mask=m, precision=precision,
                       mode=O.PLAIN if scheme == "plain" else O.ONESIDED)
    rows = sysm.nall if scheme == "plain" else sysm.nlocal
    for fused in (True, False, True):  # False: the three entry points (k_pack_count, k_pack_write)
        info = pj.compute(fused=fused)
        assert info.edge_count == count and info.edge_overflow == 0
        np.testing.assert_array_equal(canonical(*pj.edges()), canonical(s, r, m))
        assert_energy(precision, info.energy, ref["energy"], sysm.nlocal)
        assert_forces(precision, pj.forces()[:rows], ref["forces"][:rows])


@pytest.mark.parametrize("layout", ["sparse-edge", "neighbor-matrix"])
@pytest.mark.parametrize("cells", [(4, 4, 5), (21, 20, 20)])  # either side of 512 tiles
def test_float32_shell_on_the_cutoff(gpu, cells, layout):
    """One-sided float32 EAM on an undisplaced fcc lattice cut at the second-shell distance: every
    second-shell pair lies inside the float32 filter's rounding band (packed edges) or on the
    model's own float32 cutoff (matrix)."""
    a = 3.8
    box = np.array(cells, float) * a
    x = systems.wrap(systems.fcc_lattice(*cells, a), box)
    rng = np.random.default_rng(5)
    types = np.where(rng.random(len(x)) < 0.64, 1, 2).astype(np.int32)
    tables = systems.synthetic_alloy_tables(cutoff=a)
    sysm = systems.System(x, types, box, a + 1.0)
    lst = sysm.build_list(a + 1.0, kind=harness.LIST_FULL)
    pj = PairJax(sysm, ("eam", tables), precision=4, accumulation="onesided", layout=layout)
    print(f"float32 shell {layout} cells={cells} nall={sysm.nall}", flush=True)
    info = pj.compute()
    pos, sp = O.pack_atoms(sysm.x, sysm.type, sysm.nall, pj.max_atoms, 4)
    if layout == "sparse-edge":
        s, r, m, count, _ = O.pack_neighbors(sysm.x, lst, max_atoms=pj.max_atoms,
                                             max_edges=pj.max_edges, nlocal=sysm.nlocal, cutoff=a)
        assert info.edge_count == count
        np.testing.assert_array_equal(canonical(*pj.edges()), canonical(s, r, m))
    else:
        s, r, m = O.matrix_edges(*pj.neighbor_matrix(), pj.max_atoms)
    ref = O.eam_compute(tables, pos, sp, nlocal=sysm.nlocal, nghost=sysm.nghost, senders=s,
                        receivers=r, mask=m, mode=O.ONESIDED, precision=4,
                        ghost_owner=sysm.ghost_owner)
    assert_energy(4, info.energy, ref["energy"], sysm.nlocal)
    # an undisplaced alloy: forces from the two species' differences alone
    assert_forces(4, pj.forces()[:sysm.nlocal], ref["forces"][:sysm.nlocal])
