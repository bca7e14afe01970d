"""One-sided EAM steps over rows longer than the 256 slots whose validity words LDS holds.

`k_step_pack` then gives each wave whole 32-slot words and reads them back from memory for the
compacted write, at sixteen waves per 64-row tile up to 512 tiles and eight past that. Every third
row is filled with far atoms ahead of its own up to the length under test, every third cut to one
slot, and the last tile is partly filled; packed edges (float32 and, as no tile list takes such rows,
float64) and the neighbour matrix. Against the oracle: packed pairs bit for bit, forces, energy and
virial at the usual bars (lk_testutil)."""

from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from lk_testutil import assert_energy, assert_forces, assert_virial, canonical
from lammps_jax_amd import harness, systems
from lammps_jax_amd.pair import PairJax

pytestmark = pytest.mark.gpu


def _stretched(sysm, cutoff, longest):
    lst = dict(sysm.list)
    stride, rows = lst["stride"], lst["maxneighs"]
    old = np.asarray(lst["neighbors"]).reshape(rows, stride)
    num = np.array(lst["numneigh"], copy=True)
    nb = np.zeros((max(rows, longest), stride), np.int32)
    nb[:rows] = old
    rng = np.random.default_rng(3)
    pool = rng.choice(sysm.nall, 450, replace=False)
    owned = np.asarray(lst["ilist"])[:lst["inum"]]
    for i in owned[::3]:
        far = pool[np.sum((sysm.x[pool] - sysm.x[i]) ** 2, axis=1) > (cutoff + 0.1) ** 2]
        add = max(0, longest - int(num[i]))
        nb[add:add + num[i], i] = old[:num[i], i]
        nb[:add, i] = far[:add]
        num[i] += add
    num[owned[1::3]] = 1
    lst.update(neighbors=np.ascontiguousarray(nb.reshape(-1)), numneigh=num, maxneighs=len(nb))
    sysm.list = lst
    return lst


@pytest.mark.parametrize("cells", [(5, 4, 4), (21, 20, 20)])  # either side of 512 tiles
@pytest.mark.parametrize("longest", [257, 330])
@pytest.mark.parametrize("precision,layout", [(4, "sparse-edge"), (4, "neighbor-matrix"),
                                              (8, "sparse-edge"), (8, "neighbor-matrix")])
def test_long_rows(gpu, precision, layout, longest, cells):
    wl = systems.make_workload("eam_alloy_131k", cells=cells, seed=13)
    sysm = systems.System(wl.x, wl.types, wl.box, wl.cutoff + wl.skin)
    sysm.build_list(wl.cutoff + wl.skin, kind=harness.LIST_FULL)
    lst = _stretched(sysm, wl.cutoff, longest)
    pj = PairJax(sysm, ("eam", wl.tables), precision=precision, accumulation="onesided",
                 layout=layout)
    print(f"long rows {layout} precision={precision} longest={longest} nlocal={sysm.nlocal}",
          flush=True)
    pos, sp = O.pack_atoms(sysm.x, sysm.type, sysm.nall, pj.max_atoms, precision)
    nl = sysm.nlocal
    for _ in range(2):
        info = pj.compute()
        if layout == "sparse-edge":
            s, r, m, count, _ = O.pack_neighbors(sysm.x, lst, max_atoms=pj.max_atoms,
                                                 max_edges=pj.max_edges, nlocal=nl,
                                                 cutoff=wl.cutoff)
            assert info.edge_count == count and info.edge_overflow == 0
            np.testing.assert_array_equal(canonical(*pj.edges()), canonical(s, r, m))
        else:
            s, r, m = O.matrix_edges(*pj.neighbor_matrix(), pj.max_atoms)
        ref = O.eam_compute(wl.tables, pos, sp, nlocal=nl, nghost=sysm.nghost, senders=s,
                            receivers=r, mask=m, mode=O.ONESIDED, precision=precision,
                            ghost_owner=sysm.ghost_owner)
        assert_forces(precision, pj.forces()[:nl], ref["forces"][:nl])
        assert_energy(precision, info.energy, ref["energy"], nl)
        assert_virial(precision, info.virial, ref["virial"])
