"""The one-sided force sweep at every split of a tile over waves, against the oracle.

The sweep gives a 64-row tile 2, 4, 8 or 16 waves by the number of tiles (one block of sixteen
waves per CU): boxes either side of each switch on 256 CUs (256, 512 and 1,024 tiles in one
round, and more tiles than one round of two waves holds), the last tile and the last block partly
filled. Float64 at the reference's bar, float32 at 1e-5 relative (lk_testutil)."""

from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from lk_testutil import assert_energy, assert_forces, assert_virial
from lammps_jax_amd import systems
from lammps_jax_amd.pair import PairJax

pytestmark = pytest.mark.gpu

# fcc cells: tiles
BOXES = {
    "1 tile": (3, 2, 2),
    "256 tiles": (16, 16, 16),
    "257 tiles": (16, 16, 17),
    "512 tiles": (32, 16, 16),
    "526 tiles": (29, 29, 10),
    "1024 tiles": (32, 32, 16),
    "1057 tiles": (32, 32, 17),
    "2112 tiles": (33, 32, 32),
}


@pytest.mark.parametrize("precision", [8, 4])
@pytest.mark.parametrize("box", list(BOXES))
def test_force_sweep_split(gpu, box, precision):
    wl = systems.make_workload("eam_alloy_131k", cells=BOXES[box], seed=31)
    sysm = wl.system()
    lst = sysm.build_list(wl.cutoff + wl.skin)
    pj = PairJax(sysm, ("eam", wl.tables), precision=precision, accumulation="onesided")
    print(f"force split case {box} precision={precision} nlocal={sysm.nlocal}", flush=True)
    info = pj.compute()
    f = pj.forces()
    pos, sp = O.pack_atoms(sysm.x, sysm.type, sysm.nall, pj.max_atoms, precision)
    s, r, m, count, _ = O.pack_neighbors(sysm.x, lst, max_atoms=pj.max_atoms,
                                         max_edges=pj.max_edges, nlocal=sysm.nlocal,
                                         cutoff=wl.cutoff)
    ref = O.eam_compute(wl.tables, pos, sp, nlocal=sysm.nlocal, nghost=sysm.nghost, senders=s,
                        receivers=r, mask=m, mode=O.ONESIDED, ghost_owner=sysm.ghost_owner,
                        precision=precision)
    assert info.edge_count == count
    nl = sysm.nlocal
    assert_forces(precision, f[:nl], ref["forces"][:nl])
    assert np.all(f[nl:] == 0.0)
    assert_energy(precision, info.energy, ref["energy"], nl)
    assert_virial(precision, info.virial, ref["virial"])
    pj.compute(eflag=False, vflag=False)  # the sweep without the virial: the same forces
    assert np.array_equal(pj.forces(), f)
