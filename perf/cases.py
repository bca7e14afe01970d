"""The work a pair style has this library do, as timed cases.

Every case is one call that an MD engine makes on one GPU, nearly all through PairJax: the whole
force step with its result read back, the step in between outputs (forces alone, nothing read
back), the first step on a new neighbour list, the step split at the ghost exchange of a
multi-rank run, or the pack alone into the engine's own arrays. Sizes, lattices, potentials,
precisions and schemes are those of the named workloads (lammps_jax_amd.systems) and of the
benchmark, over their range of box sizes.

A case is a dict of plain values:
  model    "eam" (binary setfl alloy) or "lj" (12-6, reduced units)
  scheme   "rows" (full list, each owned row sums its own force), "half" (half list, both ends)
           or "plain" (full list, sender and receiver)
  bits     model precision, 64 or 32
  hops     receptive field in cutoffs (2: the list has ghost rows as well)
  layout   "edges" (packed edges) or "matrix" (the neighbour matrix)
  call     "step", "forces", "new_list", "exchange" or "pack"
  nx ny nz fcc cells of the box, four atoms each
  order    "lattice" (the generator's atom order) or "sorted" (the engine's spatial sort)
"""

import ctypes
import dataclasses
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "lammps-jax_amd"))

from lammps_jax_amd import _native as native  # noqa: E402
from lammps_jax_amd import harness, systems  # noqa: E402
from lammps_jax_amd.pair import DeviceComm, PairJax, contract_for  # noqa: E402

ACCUMULATION = {"rows": "onesided", "half": "half", "plain": "plain"}
EAM_A, EAM_CUTOFF, EAM_SKIN = 3.8, 6.0, 1.0
LJ_CUTOFF, LJ_SKIN = 2.5, 0.3
# neighbours of an atom in the full list (cutoff and skin) and inside the cutoff
NEIGHBORS = {"eam": (96.3, 65.2), "lj": (78.0, 54.0)}


def _case(model, scheme, bits, cells, call="step", hops=1, layout="edges", order="lattice"):
    nx, ny, nz = cells
    return dict(model=model, scheme=scheme, bits=bits, nx=nx, ny=ny, nz=nz, call=call, hops=hops,
                layout=layout, order=order)


def listed():
    named = [
        # The smallest benchmark box: a thousand LJ atoms, where launches and latency are all.
        ("lj_1k", _case("lj", "plain", 64, (8, 8, 4))),
        # The small alloy: half list, densities to both ends and folded over the ghosts.
        ("eam_8k_half", _case("eam", "half", 64, (16, 16, 8))),
        # An odd box in between thermodynamic output: forces alone, steps enqueued back to back.
        ("eam_30k_forces", _case("eam", "rows", 64, (23, 17, 19), call="forces", order="sorted")),
        # The benchmark's headline step.
        ("eam_131k", _case("eam", "rows", 64, (32, 32, 32))),
        # The same system's step right after the engine rebuilt its neighbour list.
        ("eam_131k_new_list", _case("eam", "rows", 64, (32, 32, 32), call="new_list")),
        # The step of one rank among several: density, exchange of the ghost rows, forces.
        ("eam_65k_exchange", _case("eam", "rows", 64, (32, 32, 16), call="exchange")),
        # A neighbour-matrix model at single precision, ragged box, engine-sorted atoms.
        ("eam_104k_matrix_f32", _case("eam", "rows", 32, (31, 29, 29), layout="matrix",
                                      order="sorted")),
        # The largest benchmark box: a million atoms, half list, single precision.
        ("eam_1m_half_f32", _case("eam", "half", 32, (64, 64, 64))),
        # A quarter million of them on the step that follows a list rebuild.
        ("eam_256k_half_f32_new_list", _case("eam", "half", 32, (40, 40, 40), call="new_list")),
        # LJ with a two-cutoff receptive field: rows for the ghosts too.
        ("lj_262k_hops2_f32", _case("lj", "plain", 32, (64, 32, 32), hops=2)),
        # Half that box on the step that follows a list rebuild.
        ("lj_131k_hops2_f32_new_list", _case("lj", "plain", 32, (32, 32, 32), hops=2,
                                             call="new_list")),
        # Packing alone into the caller's arrays, for an engine with its own model on the edges.
        ("pack_108k", _case("eam", "rows", 64, (30, 30, 30), call="pack")),
    ]
    return [dict(case, name=name) for name, case in named]


# What draw() picks from: model, scheme, the precisions with the most atoms of each, hops,
# layouts and calls. The least is 500 atoms everywhere.
FAMILIES = (
    ("eam", "rows", {64: 131072, 32: 131072}, (1,), ("edges", "edges", "matrix"),
     ("step", "step", "forces", "new_list", "exchange")),
    ("eam", "half", {64: 131072, 32: 1048576}, (1,), ("edges",), ("step", "forces", "new_list")),
    ("lj", "plain", {64: 131072, 32: 262144}, (1, 2), ("edges",), ("step", "forces", "new_list")),
    ("eam", "rows", {64: 131072, 32: 131072}, (1,), ("edges",), ("pack",)),
)


def draw(rng):
    model, scheme, most, hops, layouts, calls = rng.choices(FAMILIES, weights=(4, 3, 3, 1))[0]
    bits = rng.choice(sorted(most))
    atoms = math.exp(rng.uniform(math.log(500), math.log(most[bits])))
    layout, call = rng.choice(layouts), rng.choice(calls)
    if layout == "matrix" and call == "exchange":  # the exchange splits the packed-edge step
        call = "step"
    side = (atoms / 4) ** (1 / 3)
    nx = max(4, round(side * math.exp(rng.uniform(-0.3, 0.3))))
    ny = max(4, round(side * math.exp(rng.uniform(-0.3, 0.3))))
    nz = max(4, int(atoms / (4 * nx * ny)))
    return _case(model, scheme, bits, (nx, ny, nz), call=call, hops=rng.choice(hops),
                 layout=layout, order=rng.choice(("lattice", "sorted")))


def _engine(case, seed):
    """The engine's side of a step: the workload and a system with ghosts and a neighbour list."""
    cells = (case["nx"], case["ny"], case["nz"])
    base = "lj_ghost_262k" if case["model"] == "lj" else "eam_alloy_131k"
    kind = {"half": harness.LIST_HALF, "rows": harness.LIST_FULL, "plain": harness.LIST_FULL}
    wl = systems.make_workload(base, cells=cells, seed=int(seed), order=case["order"])
    wl = dataclasses.replace(
        wl, precision=case["bits"] // 8, n_hops=case["hops"],
        list_kind=harness.LIST_FULL_GHOST if case["hops"] > 1 else kind[case["scheme"]],
        accumulation=ACCUMULATION[case["scheme"]],
        edges_per_atom=96 if case["model"] == "lj" or case["bits"] == 32 else 128)
    system = wl.system()
    system.build_list(wl.cutoff + wl.skin, kind=wl.list_kind)
    return wl, system


def _prepare_pack(wl, system):
    """The pack's contract, the engine's arrays on the device and the caller's packed arrays."""
    lst, device = system.list, torch.device("cuda:0")
    max_atoms = systems.atom_capacity(system.nall)
    contract = contract_for(max_atoms=max_atoms, max_edges=max_atoms * wl.edges_per_atom,
                            cutoff=wl.cutoff, precision=wl.precision, comm=True)
    here = {k: torch.from_numpy(np.ascontiguousarray(v)).to(device)
            for k, v in (("x", system.x), ("ilist", lst["ilist"]),
                         ("numneigh", lst["numneigh"]), ("neighbors", lst["neighbors"]))}
    n = contract.max_edges
    return dict(call="pack", contract=contract, lst=lst, nlocal=system.nlocal, here=here, packed=0,
                senders=torch.full((n,), max_atoms, dtype=torch.int32, device=device),
                receivers=torch.full((n,), max_atoms, dtype=torch.int32, device=device),
                mask=torch.zeros((n,), dtype=torch.uint8, device=device),
                counts=torch.zeros((2,), dtype=torch.int32, device=device))


def prepare(case, seed):
    wl, system = _engine(case, seed)
    if case["call"] == "pack":
        return _prepare_pack(wl, system)
    layout = {"edges": "sparse-edge", "matrix": "neighbor-matrix"}[case["layout"]]
    pair = PairJax.for_workload(wl, system, layout=layout)
    state = dict(pair=pair, call=case["call"])
    if case["call"] == "exchange":
        state["comm"] = DeviceComm(pair, system)
    return state


def _run_pack(s):
    here, lst = s["here"], s["lst"]
    err = ctypes.create_string_buffer(256)
    rc = native.load().lk_pack_edges_noalloc(
        ctypes.byref(s["contract"]), torch.cuda.current_stream().cuda_stream,
        here["x"].data_ptr(), here["ilist"].data_ptr(), here["numneigh"].data_ptr(),
        here["neighbors"].data_ptr(), lst["stride"], lst["inum"], lst["gnum"], lst["maxneighs"],
        s["nlocal"], s["senders"].data_ptr(), s["receivers"].data_ptr(), s["mask"].data_ptr(),
        s["counts"].data_ptr(), s["packed"], err, len(err))
    if rc != native.LK_OK:
        raise RuntimeError(err.value.decode())
    s["packed"] = int(s["counts"][0])  # bounds the next pack's tail reset
    return {k: s[k] for k in ("senders", "receivers", "mask", "counts")}


def run(state):
    call = state["call"]
    if call == "pack":
        return _run_pack(state)
    pair = state["pair"]
    if call == "forces":
        pair.enqueue(eflag=False, vflag=False)
        return dict(f=pair.f)
    if call == "exchange":
        info = pair.compute_split(state["comm"], fused=True)
    else:
        if call == "new_list":  # the engine's rebuild signal
            pair.list_epoch += 1
            pair.h.set_list_epoch(pair.list_epoch)
        info = pair.compute()
    return dict(f=pair.f, energy=info.energy, virial=info.virial)


def _sizes(case):
    """(owned atoms, owned and ghost atoms, list rows, list entries, packed edges), from the
    densities."""
    a = EAM_A if case["model"] == "eam" else systems.lj_lattice_constant()
    cutoff, skin = (EAM_CUTOFF, EAM_SKIN) if case["model"] == "eam" else (LJ_CUTOFF, LJ_SKIN)
    box = [a * case[k] for k in ("nx", "ny", "nz")]
    shell = case["hops"] * cutoff + skin
    owned = 4 * case["nx"] * case["ny"] * case["nz"]
    atoms = 4 / a ** 3 * math.prod(side + 2 * shell for side in box)
    # with a two-cutoff field the ghosts have rows too, those at the rim shorter ones
    rows = owned if case["hops"] == 1 else 0.96 * atoms
    in_list, packed = NEIGHBORS[case["model"]]
    share = 0.5 if case["scheme"] == "half" else 1.0
    return owned, atoms, rows, rows * share * in_list, rows * share * packed


def work(case):
    owned, atoms, rows, entries, edges = _sizes(case)
    held = atoms if case["scheme"] != "rows" else owned  # rows of f that change
    # list and positions in, packed edges out (a matrix step packs none), forces in and out
    nbytes = 4 * entries + 8 * rows + 28 * atoms
    if case["layout"] == "edges":
        nbytes += 9 * edges
    if case["call"] == "pack":
        return dict(bytes=nbytes, flops=8 * entries)
    # per packed edge: LJ energy and force 30; EAM density 20 and force 50 for each end
    per_edge = 30 if case["model"] == "lj" else (140 if case["scheme"] == "half" else 70)
    return dict(bytes=nbytes + 48 * held, flops=8 * entries + per_edge * edges)


def tolerance(case):
    if case["call"] == "pack":
        return "exact"
    # 64 bits: forces come within 2e-15 of `exact` and virials near zero pressure within 5e-14.
    # 32 bits: 1e-5 to 5e-5, most of it positions rounded to 32 bits.
    return {"rel": 1e-12} if case["bits"] == 64 else {"rel": 1e-4}


# ---------------------------------------------------------------------------------------------
# The same results in 64 bits with plain torch
# ---------------------------------------------------------------------------------------------
def _pairs(system, lst, cutoff, rows, device, chunk):
    """Chunks of the list's (i, j) inside the cutoff with i among the first `rows` atoms."""
    x = torch.from_numpy(system.x).to(device)
    ilist = torch.from_numpy(lst["ilist"]).to(device).long()
    ilist = ilist[ilist < rows]
    num = torch.from_numpy(lst["numneigh"]).to(device).long()
    neighbors = torch.from_numpy(lst["neighbors"]).to(device)
    neighbors = neighbors.view(lst["maxneighs"], lst["stride"])
    step = max(1, chunk // max(1, len(ilist)))
    for lo in range(0, lst["maxneighs"], step):
        slots = torch.arange(lo, min(lo + step, lst["maxneighs"]), device=device)
        j = neighbors[slots[:, None], ilist[None, :]].long() & 0x3FFFFFFF
        i = ilist[None, :].expand_as(j)
        have = slots[:, None] < num[ilist][None, :]
        i, j = i[have], j[have]
        d = x[j] - x[i]
        r2 = (d * d).sum(1)
        keep = r2 < cutoff * cutoff
        yield i[keep], j[keep], d[keep], r2[keep].sqrt()


def _spline(coef, table, x, step):
    """Value and slope of spline `table` (a row of coef [tables][nodes][4]) at x."""
    n = coef.shape[1]
    at = x / step
    node = at.floor().clamp(0, n - 2)
    t = (at - node).clamp(max=1.0)
    c = coef[table, node.long()]
    value = c[:, 0] + t * (c[:, 1] + t * (c[:, 2] + t * c[:, 3]))
    slope = (c[:, 1] + t * (2 * c[:, 2] + 3 * t * c[:, 3])) / step
    return value, slope


def exact(case, seed):
    if case["call"] == "pack":
        return None
    device = torch.device("cuda:0" if torch.cuda.is_available() else "cpu")
    wl, system = _engine(case, seed)
    lst, nlocal, nall = system.list, system.nlocal, system.nall
    f64 = dict(dtype=torch.float64, device=device)
    x = torch.from_numpy(system.x).to(device)
    f = torch.zeros((nall, 3), **f64)
    both = case["scheme"] != "rows"  # receivers take the opposite force
    energy = torch.zeros((), **f64)
    pair_virial = torch.zeros((3, 3), **f64)
    chunk = 1 << 22

    def add(i, j, coef, d):
        nonlocal pair_virial
        g = coef[:, None] * d
        f.index_add_(0, i, g)
        if both:
            f.index_add_(0, j, -g)
        else:
            pair_virial = pair_virial - 0.5 * (g.T @ d)

    if case["model"] == "lj":
        eps, sig, half = wl.lj["epsilon"], wl.lj["sigma"], wl.lj["edge_energy_scale"]
        for i, j, d, r in _pairs(system, lst, wl.cutoff, nlocal, device, chunk):
            u = (sig / r) ** 6
            energy += (half * 4 * eps * (u * u - u)).sum()
            add(i, j, -half * 4 * eps * (12 * u * u - 6 * u) / (r * r), d)
    else:
        tab = {k: torch.from_numpy(np.ascontiguousarray(wl.tables[k])).to(device)
               for k in ("embedding", "density", "pair")}
        dr, drho = wl.tables["dr"], wl.tables["drho"]
        species = torch.from_numpy(system.type).to(device).long() - 1
        owner = torch.arange(nall, device=device)
        owner[nlocal:] = torch.from_numpy(system.ghost_owner).to(device).long()
        rho = torch.zeros(nall, **f64)
        for i, j, d, r in _pairs(system, lst, wl.cutoff, nlocal, device, chunk):
            rho.index_add_(0, owner[i], _spline(tab["density"], species[j], r, dr)[0])
            if both:
                rho.index_add_(0, owner[j], _spline(tab["density"], species[i], r, dr)[0])
        value, slope = _spline(tab["embedding"], species[:nlocal], rho[:nlocal], drho)
        energy += value.sum()
        fp = slope[owner]
        for i, j, d, r in _pairs(system, lst, wl.cutoff, nlocal, device, chunk):
            hi, lo = torch.maximum(species[i], species[j]), torch.minimum(species[i], species[j])
            z, zp = _spline(tab["pair"], hi * (hi + 1) // 2 + lo, r, dr)
            phi = z / r
            energy += (1.0 if both else 0.5) * phi.sum()
            psip = (fp[i] * _spline(tab["density"], species[j], r, dr)[1]
                    + fp[j] * _spline(tab["density"], species[i], r, dr)[1] + (zp - phi) / r)
            add(i, j, psip / r, d)
    if case["call"] == "forces":
        return dict(f=f)
    w = f.T @ x if both else pair_virial  # f.r over all rows, or the pair sum of whole rows
    virial = torch.stack([w[0, 0], w[1, 1], w[2, 2], w[1, 0], w[2, 0], w[2, 1]])
    return dict(f=f, energy=float(energy), virial=virial)
