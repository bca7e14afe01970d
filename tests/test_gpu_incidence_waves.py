"""The incidence build at each split of a 64-row tile over its counting waves (2, 4, 8 or 16 by the
number of tiles: switches at 64, 512 and 2,048 tiles on 256 CUs), against the oracle, and a rebuild of
the same list with the first build bit for bit. Float64: forces and virials at the reference's
bar (lk_testutil)."""

from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from lk_testutil import assert_forces, assert_virial
from lammps_jax_amd import harness, systems
from lammps_jax_amd.pair import PairJax

pytestmark = pytest.mark.gpu

# scheme, fcc cells (64-row tiles)
CASES = [("plain", (16, 16, 4)), ("half", (13, 10, 8)), ("half", (32, 16, 16)),
         ("plain", (27, 19, 16)), ("plain", (32, 32, 32)), ("half", (33, 32, 32))]


@pytest.mark.parametrize("scheme,cells", CASES)
def test_incidence_waves(gpu, scheme, cells):
    half = scheme == "half"
    wl = systems.make_workload("eam_alloy_8k" if half else "lj_ghost_262k", cells=cells, seed=6)
    sysm = systems.System(wl.x, wl.types, wl.box, wl.cutoff + wl.skin)
    sysm.build_list(wl.cutoff + wl.skin, kind=harness.LIST_HALF if half else harness.LIST_FULL)
    model = ("eam", wl.tables) if half else ("lj", wl.lj)
    pj = PairJax(sysm, model, precision=8, accumulation=scheme, fused=True)
    print(f"incidence waves {scheme} cells={cells} nlocal={sysm.nlocal}", flush=True)
    info = pj.compute()
    f = pj.forces().copy()
    pj.list_epoch += 1  # the engine's rebuild signal: the same lists again
    pj.h.set_list_epoch(pj.list_epoch)
    again = pj.compute()
    assert again.energy == info.energy
    assert np.array_equal(pj.forces(), f)
    pos, sp = O.pack_atoms(sysm.x, sysm.type, sysm.nall, pj.max_atoms, 8)
    s, r, m, count, _ = O.pack_neighbors(sysm.x, sysm.list, max_atoms=pj.max_atoms,
                                         max_edges=pj.max_edges, nlocal=sysm.nlocal,
                                         cutoff=wl.cutoff)
    kw = dict(nlocal=sysm.nlocal, nghost=sysm.nghost, senders=s, receivers=r, mask=m, precision=8)
    if half:
        ref = O.eam_compute(wl.tables, pos, sp, ghost_owner=sysm.ghost_owner, mode=O.HALF, **kw)
    else:
        ref = O.lj_compute(wl.lj, pos, mode=O.PLAIN, **kw)
    nall = sysm.nall
    assert info.edge_count == count
    # The oracle adds the edges' energies one after another: each of the `count` additions rounds
    # the running sum by at most 2^-53 of it, signs at random, so the sum is off by about
    # sqrt(count) 2^-53 |E| (2.6e-7 of the 131,072 LJ atoms' 8.8e5, where 1e-13 per atom is 1.3e-8).
    bar = max(1e-13 * sysm.nlocal, np.sqrt(count) * 2.0 ** -53 * abs(ref["energy"]))
    assert abs(info.energy - ref["energy"]) <= bar, (info.energy, ref["energy"])
    assert_forces(8, f[:nall], ref["forces"][:nall])
    assert_virial(8, info.virial, O.virial_fdotr(ref["forces"][:nall], sysm.x, nall))
