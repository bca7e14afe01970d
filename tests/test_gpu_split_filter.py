"""Float32 sweeps after a pack called on its own, with a neighbour shell on the cutoff.

Inside the rounding band of the cutoff the sweeps take the pack's own decision, from its validity
bits. The engine's list is theirs to read until the calls that build the incidence lists from it,
and no longer: on later steps of the same list its arrays may change once lk_pack_edges has been
called, also where the lists were built by the fused step, which needs no bits. The engine here
overwrites them (with other valid entries) between the pack and the model pass. A perturbed lattice
cut at its second-shell distance, so that about half of that shell is kept and float32 decides none
of it: rows as the list has them, rows made longer by far atoms (bins of fewer atoms, and bins whose
entries are sorted) and rows that name some of the shell twice. Against the oracle, and each step with
the first bit for bit."""

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


def _longer(sysm, longest, twice):
    """The list with every third row filled up to `longest` slots by atoms past the cutoff, ahead of
    its own, and with `twice` half the rows naming one of their neighbours again."""
    lst = dict(sysm.list)
    stride, rows = lst["stride"], lst["maxneighs"]
    old = np.asarray(lst["neighbors"]).reshape(rows, stride) & 0x3FFFFFFF
    num = np.array(lst["numneigh"], copy=True)
    nb = np.zeros((max(rows + 1, longest), stride), np.int32)
    nb[:rows] = old
    x = sysm.x[:sysm.nall]
    rng = np.random.default_rng(9)
    for n, i in enumerate(np.asarray(lst["ilist"])[:lst["inum"]]):
        own = old[:num[i], i]
        if twice and n % 2 and len(own):
            own = np.insert(own, rng.integers(0, len(own) + 1), rng.choice(own))
        far = np.flatnonzero(np.sum((x - x[i]) ** 2, axis=1) > (A + 0.1) ** 2)
        add = np.resize(far, max(0, longest - len(own)) if n % 3 == 0 else 0)
        num[i] = len(add) + len(own)
        nb[:num[i], i] = np.concatenate([add, own])
    lst.update(neighbors=np.ascontiguousarray(nb.reshape(-1)), numneigh=num, maxneighs=len(nb))
    sysm.list = lst
    return lst


@pytest.mark.parametrize("first", ["fused", "split"])
@pytest.mark.parametrize("scheme,cells,longest,twice", [
    ("half", (5, 5, 5), 0, False), ("half", (9, 8, 8), 0, False), ("plain", (5, 5, 5), 0, False),
    ("plain lj", (9, 8, 7), 0, False), ("half", (5, 5, 5), 300, False),
    ("plain", (4, 5, 5), 200, False), ("half", (5, 4, 5), 1700, False),
    ("plain lj", (5, 5, 4), 1500, False), ("plain lj", (5, 5, 5), 0, True),
    ("half", (5, 5, 5), 0, True), ("plain", (5, 4, 5), 1500, True)])
def test_split_steps_on_a_standing_list(gpu, scheme, cells, longest, twice, first):
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
    if longest or twice:
        lst = _longer(sysm, longest, twice)
    pj = PairJax(sysm, model, precision=4, accumulation=scheme.split()[0])
    nl, nall = sysm.nlocal, sysm.nall
    print(f"split filter {scheme} cells={cells} room={lst['maxneighs']} first={first} nall={nall}",
          flush=True)
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
