"""The list-built incidence lists of the two-sided schemes at the edges of their binned build.

The build brings each bin's entries (the slots naming its atoms) together in LDS: 64 atoms to a bin,
fewer where the list's room asks for it; past 218 slots of room (`maxneighs` is padded here, as an
engine's list may be) it measures the rows first and goes by the longest. Bins that more entries name
than LDS holds sort them (every row given far atoms of one bin, which the cutoff drops again; in the
plain scheme they have no reverse). Rows that are long themselves: test_gpu_incidence_room.py and
test_gpu_incidence_repeats.py. Each is compared with the oracle, and a rebuild of the same list with
the first build bit for bit."""

from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from lk_testutil import assert_energy, assert_forces, assert_virial
from lammps_jax_amd import harness, systems
from lammps_jax_amd.pair import PairJax

pytestmark = pytest.mark.gpu


def _edited(sysm, wl, width, hubs):
    """The system's list with `width` slots of room per row and `hubs` far atoms appended to the
    slots of each owned row (those of the first hubs atoms that lie past the cutoff and are not
    in the row)."""
    lst = dict(sysm.list)
    stride, rows = lst["stride"], lst["maxneighs"]
    nb = np.asarray(lst["neighbors"]).reshape(rows, stride)
    num = np.array(lst["numneigh"], copy=True)
    room = max(width, rows + hubs)
    wide = np.zeros((room, stride), np.int32)
    wide[:rows] = nb
    if hubs:
        x = sysm.x[:sysm.nall]
        for i in np.asarray(lst["ilist"])[:lst["inum"]]:
            have = set((wide[:num[i], i] & 0x3FFFFFFF).tolist())
            far = np.sum((x[:hubs] - x[i]) ** 2, axis=1) > (wl.cutoff + 0.1) ** 2
            for j in range(hubs):
                if far[j] and j not in have:
                    wide[num[i], i] = j
                    num[i] += 1
    lst.update(neighbors=np.ascontiguousarray(wide.reshape(-1)), numneigh=num, maxneighs=room)
    sysm.list = lst
    return lst


CASES = [  # scheme, precision, cells, width, hubs
    ("plain", 8, (4, 4, 4), 0, 0),
    ("plain", 4, (5, 4, 4), 240, 0),
    ("plain", 8, (4, 4, 4), 1800, 0),
    ("plain", 4, (7, 7, 7), 0, 1),
    ("half", 8, (4, 5, 4), 0, 0),
    ("half", 4, (4, 4, 4), 700, 0),
    ("half", 4, (4, 4, 4), 1800, 0),
    ("half", 8, (9, 8, 8), 0, 12),
]


@pytest.mark.parametrize("scheme,precision,cells,width,hubs", CASES)
def test_binned_incidence_lists(gpu, scheme, precision, cells, width, hubs):
    half = scheme == "half"
    wl = systems.make_workload("eam_alloy_8k" if half else "lj_ghost_262k", cells=cells, seed=5)
    hops = 1 if half else 2
    sysm = systems.System(wl.x, wl.types, wl.box, hops * wl.cutoff + wl.skin)
    sysm.build_list(wl.cutoff + wl.skin,
                    kind=harness.LIST_HALF if half else harness.LIST_FULL_GHOST)
    lst = _edited(sysm, wl, width, hubs)
    model = ("eam", wl.tables) if half else ("lj", wl.lj)
    pj = PairJax(sysm, model, precision=precision, accumulation=scheme, n_hops=hops, fused=True)
    print(f"incidence bins {scheme} precision={precision} cells={cells} width={lst['maxneighs']} "
          f"hubs={hubs} nall={sysm.nall}", flush=True)
    info = pj.compute()
    f = pj.forces().copy()
    pos, sp = O.pack_atoms(sysm.x, sysm.type, sysm.nall, pj.max_atoms, precision)
    s, r, m, count, _ = O.pack_neighbors(sysm.x, lst, max_atoms=pj.max_atoms,
                                         max_edges=pj.max_edges, nlocal=sysm.nlocal,
                                         cutoff=wl.cutoff, n_hops=hops)
    kw = dict(nlocal=sysm.nlocal, nghost=sysm.nghost, senders=s, receivers=r, mask=m,
              precision=precision, owned_rows_only=True)
    if half:
        ref = O.eam_compute(wl.tables, pos, sp, ghost_owner=sysm.ghost_owner, mode=O.HALF, **kw)
    else:
        ref = O.lj_compute(wl.lj, pos, mode=O.PLAIN, **kw)
    nall = sysm.nall
    assert info.edge_count == count
    assert_energy(precision, info.energy, ref["energy"], sysm.nlocal)
    assert_forces(precision, f[:nall], ref["forces"][:nall])
    assert_virial(precision, info.virial, O.virial_fdotr(ref["forces"][:nall], sysm.x, nall))
    pj.list_epoch += 1  # the engine's rebuild signal: the same lists again
    pj.h.set_list_epoch(pj.list_epoch)
    again = pj.compute()
    assert again.energy == info.energy
    assert np.array_equal(pj.forces(), f)
