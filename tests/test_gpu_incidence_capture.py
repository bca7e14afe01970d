"""A list rebuild under graph capture: the incidence build neither allocates nor waits.

The build's working arrays are sized by the contract's capacity, so a list with room for longer rows
than any before (its bins smaller and more of them) can be built inside a captured step once the
validity bits have been sized for it. Replays, with eager steps on either list and synchronizations
between them, give the eager step's forces bit for bit."""

from __future__ import annotations

import numpy as np
import pytest

from lammps_jax_amd import harness, systems
from lammps_jax_amd.pair import PairJax

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme,precision", [("plain", 4), ("half", 8)])
def test_rebuild_with_more_room_under_capture(gpu, scheme, precision):
    import torch

    half = scheme == "half"
    wl = systems.make_workload("eam_alloy_8k" if half else "lj_ghost_262k", cells=(5, 4, 4), seed=3)
    sysm = systems.System(wl.x, wl.types, wl.box, wl.cutoff + wl.skin)
    tight = sysm.build_list(wl.cutoff + wl.skin,
                            kind=harness.LIST_HALF if half else harness.LIST_FULL)
    room = 400
    nb = np.zeros((room, tight["stride"]), np.int32)
    nb[:tight["maxneighs"]] = np.asarray(tight["neighbors"]).reshape(-1, tight["stride"])
    wide = dict(tight, neighbors=nb.reshape(-1), maxneighs=room)
    model = ("eam", wl.tables) if half else ("lj", wl.lj)
    # edge capacity of half the wide list's slots at least: the entries' arrays hold either list
    pj = PairJax(sysm, model, precision=precision, accumulation=scheme,
                 max_edges=tight["inum"] * room)
    neighbors = {id(lst): torch.from_numpy(lst["neighbors"]).to(pj.device) for lst in (tight, wide)}

    def use(lst):
        sysm.list = lst
        pj.neighbors = neighbors[id(lst)]
        pj.list_epoch += 1
        pj.h.set_list_epoch(pj.list_epoch)

    def eager(lst):
        use(lst)
        pj.enqueue(vflag=False)
        return pj.forces().copy()

    print(f"capture {scheme} precision={precision} room {tight['maxneighs']} -> {room}", flush=True)
    use(wide)
    pj.pack()  # sizes the validity bits
    want = eager(tight)
    assert np.abs(want).max() > 0
    use(wide)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        pj.enqueue(vflag=False)
    for lst in (None, tight, wide, tight):
        if lst is not None:
            assert np.array_equal(eager(lst), want)
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(pj.forces(), want)
