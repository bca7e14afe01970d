"""Float32 sweeps after a pack called on its own, with a neighbour shell on the cutoff.

Inside the rounding band of the cutoff the sweeps take the pack's own decision, from its validity
bits. The engine's list is theirs to read until the calls that build the incidence lists from it,
and no longer: on later steps of the same list its arrays may change once lk_pack_edges has been
called, also where the lists were built by the fused step, which needs no bits. The engine here
overwrites them (with other valid entries) between the pack and the model pass. A perturbed lattice
cut at its second-shell distance, so that about half of that shell is kept and float32 decides none
of it. Against the oracle, and each step with the first bit for bit."""

from __future__ import annotations

import numpy as np
import pytest

import oracle as O
from lk_testutil import assert_energy, assert_forces, canonical
from lammps_jax_amd import harness, systems
from lammps_jax_amd.pair import DeviceComm, PairJax

pytestmark = pytest.mark.gpu

A = 3.8


class _Overwriting(DeviceComm):
    """Exchanges that find the engine's list overwritten."""

    def forward(self, rows, width):
        _overwrite(self.pair)
        super().forward(rows, width)


def _overwrite(pj):
    pj.neighbors.zero_()
    pj.numneigh.fill_(1)
    pj.ilist.zero_()


def _split(pj):
    s, lst, st = pj.system, pj.system.list, pj.stream()
    pj.f.zero_()
    pj.h.pack_atoms(st, pj.x.data_ptr(), pj.type.data_ptr(), s.nall)
    pj.h.pack_edges(st, pj.x.data_ptr(), pj.ilist.data_ptr(), pj.numneigh.data_ptr(),
                    pj.neighbors.data_ptr(), lst["stride"], lst["inum"], lst["gnum"],
                    lst["maxneighs"], s.nlocal)
    _overwrite(pj)
    pj.h.compute(st, s.nlocal, s.nghost, 1, pj.scale, pj.f.data_ptr())
    return pj.h.step_result(st)


@pytest.mark.parametrize("first", ["fused", "split"])
@pytest.mark.parametrize("scheme,cells", [("half", (5, 5, 5)), ("half", (9, 8, 8)),
                                          ("plain", (5, 5, 5)), ("plain lj", (9, 8, 7))])
def test_split_steps_on_a_standing_list(gpu, scheme, cells, first):
    half, lj = scheme == "half", scheme.endswith("lj")
    box = np.array(cells, float) * A
    rng = np.random.default_rng(5)
    x = systems.fcc_lattice(*cells, A)
    x = systems.wrap(x + rng.uniform(-1e-6, 1e-6, size=x.shape), box)
    types = np.where(rng.random(len(x)) < 0.64, 1, 2).astype(np.int32)
    if lj:
        model = ("lj", dict(epsilon=1.0, sigma=2.4, cutoff=A, edge_energy_scale=0.5))
    else:
        model = ("eam", systems.synthetic_alloy_tables(cutoff=A))
    sysm = systems.System(x, types, box, A + 1.0)
    lst = sysm.build_list(A + 1.0, kind=harness.LIST_HALF if half else harness.LIST_FULL)
    pj = PairJax(sysm, model, precision=4, accumulation=scheme.split()[0])
    nl, nall = sysm.nlocal, sysm.nall
    print(f"split filter {scheme} cells={cells} first={first} nall={nall}", flush=True)
    pos, sp = O.pack_atoms(sysm.x, sysm.type, nall, pj.max_atoms, 4)
    s, r, m, count, _ = O.pack_neighbors(sysm.x, lst, max_atoms=pj.max_atoms,
                                         max_edges=pj.max_edges, nlocal=nl, cutoff=A)
    kw = dict(nlocal=nl, nghost=sysm.nghost, senders=s, receivers=r, mask=m, precision=4,
              mode=O.HALF if half else O.PLAIN)
    if lj:
        ref = O.lj_compute(model[1], pos, **kw)
    else:
        ref = O.eam_compute(model[1], pos, sp, ghost_owner=sysm.ghost_owner, **kw)
    info = pj.compute(fused=first == "fused")
    want = pj.forces().copy()
    assert info.edge_count == count
    np.testing.assert_array_equal(canonical(*pj.edges()), canonical(s, r, m))
    assert_energy(4, info.energy, ref["energy"], nl)
    assert_forces(4, want[:nall], ref["forces"][:nall])
    saved = [t.clone() for t in (pj.ilist, pj.numneigh, pj.neighbors)]
    for _ in range(2):
        again = _split(pj)
        assert again.energy == info.energy
        assert np.array_equal(pj.forces(), want)
        for t, old in zip((pj.ilist, pj.numneigh, pj.neighbors), saved):
            t.copy_(old)
    if half:  # the pass split at its exchanges
        pj.compute_split(_Overwriting(pj, sysm))
        # the exchange sums the ghost densities in another order than the single-rank fold
        assert_forces(4, pj.forces()[:nall], ref["forces"][:nall])
