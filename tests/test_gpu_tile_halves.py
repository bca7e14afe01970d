"""The tile step with a block per 64-row half of a tile, against the oracle.

Up to one 128-row tile per CU (256 tiles) each half of a tile has a block of its own; past that a
block takes a whole tile. Boxes of one row tile (its second half empty, and one row into it), of a
partly filled last half, and either side of the switch, for both densities' steps: the whole step and
the one split at the exchange. Float64 at the reference's bar (lk_testutil)."""

from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from lk_testutil import assert_energy, assert_forces, assert_virial, canonical
from lammps_jax_amd import systems
from lammps_jax_amd.pair import DeviceComm, PairJax

pytestmark = pytest.mark.gpu

BOXES = {"48 rows": (3, 2, 2), "64 rows": (4, 2, 2), "72 rows": (3, 3, 2), "252 rows": (7, 3, 3),
         "32768 rows": (32, 16, 16), "32816 rows": (14, 293, 2)}


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("box", list(BOXES))
def test_tile_halves(gpu, box, split):
    cells = BOXES[box]
    wl = systems.make_workload("eam_alloy_131k", cells=cells, seed=37)
    sysm = wl.system()
    lst = sysm.build_list(wl.cutoff + wl.skin)
    pj = PairJax(sysm, ("eam", wl.tables), precision=8, accumulation="onesided")
    print(f"tile halves {box} split={split} nlocal={sysm.nlocal}", flush=True)
    pos, sp = O.pack_atoms(sysm.x, sysm.type, sysm.nall, pj.max_atoms, 8)
    s, r, m, count, _ = O.pack_neighbors(sysm.x, lst, max_atoms=pj.max_atoms,
                                         max_edges=pj.max_edges, nlocal=sysm.nlocal,
                                         cutoff=wl.cutoff)
    ref = O.eam_compute(wl.tables, pos, sp, nlocal=sysm.nlocal, nghost=sysm.nghost, senders=s,
                        receivers=r, mask=m, mode=O.ONESIDED, ghost_owner=sysm.ghost_owner,
                        precision=8)
    nl = sysm.nlocal
    for _ in range(2):
        info = (pj.compute_split(DeviceComm(pj, sysm), fused=True) if split else pj.compute())
        assert info.edge_count == count and info.edge_overflow == 0
        np.testing.assert_array_equal(canonical(*pj.edges()), canonical(s, r, m))
        assert_forces(8, pj.forces()[:nl], ref["forces"][:nl])
        assert_energy(8, info.energy, ref["energy"], nl)
        assert_virial(8, info.virial, ref["virial"])
