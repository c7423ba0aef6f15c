"""Performance cases of the erdst hot path: what a user's erdst run asks of
the library, through the ctypes binding of its C ABI.

A block case is one averaging block of a run: clear the accumulators, give
the library every frame (and, in refs runs, its insertions), run it, and
fetch the block's distributions -- the loop of `python -m erdst_gpu.erdst`.
An energies case runs one frame and reads the per-(insertion, molecule)
energies instead, as a program does that bins or reweights them itself.  (A
block's counts turn on the last bit of an energy at a bin edge, so the two
kinds are compared differently: the distributions value for value, the
energies as floats.)

`exact` forms the same outputs in 64 bits from the same inputs: every site
pair by brute force, and the particle-mesh sum with the spread, the FFT and
the gather of each insertion written out.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ermod-openacc_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from erdst_gpu import capi, synth  # noqa: E402
from erdst_gpu.params import hot_path_params  # noqa: E402
from erdst_gpu.topology import Species, build_topology  # noqa: E402

# What a case's values mean: mode refs or soln; the solvent (rigid 3-site
# waters, rigid chains of chain_sites sites); the solutes of a refs run (the
# largest has `sites` sites, the others fewer, spread over the logarithm), or
# the one solute of a soln run; nins insertions per solute and frame; frames
# per block; the orthorhombic box lx ly lz, skewed when tilt; the PME grid and
# spline order; cltype 2 PME, 0 bare Coulomb; bins of the energy mesh per
# species; corr: form ecorr; host: inputs in host memory (a trajectory
# reader's), else resident on the GPU; graph: the block's frames recorded
# once as a HIP graph and replayed.  layout: mixed (solvent everywhere), slab
# (chains between water, insertions among the chains), vapour (a liquid film,
# insertions in the gap above it).
_BASE = dict(mode="refs", waters=1000, chains=0, chain_sites=50, solutes=1, sites=5, flex=True, nins=100, frames=1,
             lx=31.04, ly=31.04, lz=31.04, tilt=False, layout="mixed", ms1=32, ms2=32, ms3=32, order=4, cltype=2,
             bins=600, corr=True, host=False, graph=False, out="block")


def _case(name=None, **kw):
    c = dict(_BASE, **kw)
    if name is not None:
        c["name"] = name
    return c


def _cube(L):
    return dict(lx=L, ly=L, lz=L)


def _grid(*k):
    k = k * 3 if len(k) == 1 else k
    return dict(ms1=k[0], ms2=k[1], ms3=k[2])


def listed():
    return [
        # the smallest call: a few insertions into a box just above the cutoff, inputs from the host,
        # the reference's default spline order; latency and launches are all of it
        _case("refs_tiny", waters=517, **_cube(24.9), **_grid(32), order=6, nins=7, bins=240, host=True),
        # a small refs run: 1000 waters, 100 insertions per frame, ten frames per block
        _case("refs_1k", nins=100, frames=10),
        # the same kind of run for production sampling: the block's frames recorded as one graph
        _case("refs_2k_graph", waters=2000, **_cube(39.1), **_grid(40), order=6, nins=96, frames=8, flex=False,
              graph=True),
        # a solution run, one flexible 20-site solute in 8000 waters, distributions and correlations,
        # frames as a trajectory reader delivers them
        _case("soln_8k", mode="soln", waters=8000, **_cube(62.1), **_grid(64), sites=20, bins=1200, frames=6, host=True),
        # a solution run of a large solute at the default order, no correlations (erdst's default for soln)
        _case("soln_large_solute", mode="soln", waters=12001, **_cube(72.4), **_grid(72), order=6, sites=150, bins=1200,
              frames=5, corr=False, host=True),
        # the main workload: 30 000 waters, 1000 insertions per frame
        _case("refs_90k", waters=30000, **_cube(67.0), **_grid(72), nins=1000, frames=3),
        # the same box at the reference's default spline order, a ragged number of insertions, rigid solute
        _case("refs_90k_order6", waters=30000, **_cube(67.0), **_grid(72), order=6, nins=700, frames=2, flex=False),
        # several solutes in one context over a two-species solvent, 1 to 45 sites
        _case("refs_8_solutes", waters=12000, chains=2000, chain_sites=9, **_cube(80.0), **_grid(80), solutes=8,
              sites=45, nins=250, frames=2, flex=False, bins=300),
        # the largest: 200 000 atoms, a polymer slab between water, a flexible 150-site solute
        _case("refs_slab_200k", waters=16667, chains=3000, lx=120.0, ly=120.0, lz=100.0, layout="slab",
              **_grid(128, 128, 108), sites=150, nins=256, frames=2),
        # energies of insertions above a polymer film: a non-cubic box, grid lengths as the box's sides ask for them
        _case("film_energies", waters=1200, chains=500, lx=58.0, ly=58.0, lz=96.0, layout="vapour",
              **_grid(60, 60, 100), order=6, sites=9, nins=300, out="energies"),
        # the same with a larger solute, order 5 and odd sizes everywhere, inputs from the host
        _case("film_energies_odd", waters=777, chains=191, chain_sites=37, lx=45.0, ly=49.0, lz=73.0, layout="vapour",
              **_grid(45, 50, 75), order=5, sites=25, nins=101, out="energies", host=True),
        # bare Coulomb in a skewed cell: the pair search, the binning and the correlations alone
        _case("refs_bare_skewed", waters=9001, **_cube(64.6), tilt=True, cltype=0, nins=333, frames=3),
    ]


_SQUARE = [32, 36, 40, 48, 64, 72, 80, 96]     # grid lengths that are common in use
_ANY = [45, 50, 54, 60, 64, 75, 80, 90, 96, 100, 108]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["small", "refs", "refs", "soln", "several", "slab", "film", "film", "bare"])
    order = rng.choice([4, 4, 6, 6, 5])
    host, flex = rng.random() < 0.5, rng.random() < 0.7
    if kind in ("small", "refs"):
        waters = _log(rng, 517, 3000) if kind == "small" else _log(rng, 3000, 30000)
        L = round((waters * 29.9) ** (1 / 3) + rng.uniform(0.0, 1.0), 2)
        nins = _log(rng, 7, 120) if kind == "small" else _log(rng, 60, 1000)
        K = min(_SQUARE, key=lambda k: abs(k - L * rng.uniform(0.95, 1.15)))
        frames = rng.randint(1, 6) if kind == "small" else rng.randint(1, 3)
        graph = kind == "small" and not host and rng.random() < 0.5
        return _case(waters=waters, **_cube(L), **_grid(K), order=order, nins=nins, frames=frames, flex=flex,
                     sites=rng.choice([1, 3, 5, 7, 11, 16]), bins=rng.choice([240, 450, 600]), host=host, graph=graph)
    if kind == "soln":
        waters = _log(rng, 2000, 16000)
        L = round((waters * 30.5) ** (1 / 3) + 1.0, 2)
        K = min(_SQUARE, key=lambda k: abs(k - L * rng.uniform(0.95, 1.15)))
        return _case(mode="soln", waters=waters, **_cube(L), **_grid(K), order=order, sites=_log(rng, 5, 120),
                     bins=1200, frames=rng.randint(1, 6), corr=rng.random() < 0.5, host=True)
    if kind == "several":
        waters = _log(rng, 4000, 12000)
        chains = waters // 8
        L = round((waters * 29.9 + chains * 75.0) ** (1 / 3), 2)
        K = min(_SQUARE, key=lambda k: abs(k - L * rng.uniform(0.95, 1.1)))
        return _case(waters=waters, chains=chains, chain_sites=9, **_cube(L), **_grid(K), order=order,
                     solutes=rng.randint(2, 8), sites=_log(rng, 5, 45), nins=_log(rng, 40, 400), flex=False, bins=300)
    if kind == "slab":
        chains = _log(rng, 300, 2000)
        a = round((chains * 50 * 5.0 / 40.0) ** 0.5 + 30.0, 1)
        K = min(_SQUARE, key=lambda k: abs(k - a))
        return _case(waters=_log(rng, 1500, 8000), chains=chains, lx=a, ly=a, lz=100.0, layout="slab",
                     **_grid(K), order=4, sites=_log(rng, 13, 150), nins=_log(rng, 30, 200), host=host)
    if kind == "film":
        a, b = round(rng.uniform(40.0, 62.0), 1), round(rng.uniform(40.0, 62.0), 1)
        c = round(rng.uniform(70.0, 98.0), 1)
        k = [min(_ANY, key=lambda k: abs(k - s * rng.uniform(0.9, 1.1))) for s in (a, b, c)]
        return _case(waters=_log(rng, 300, 1500), chains=_log(rng, 80, 300), chain_sites=rng.randint(12, 50), lx=a,
                     ly=b, lz=c, layout="vapour", **_grid(*k), order=order, sites=_log(rng, 3, 30),
                     nins=_log(rng, 17, 300), out="energies", host=host)
    waters = _log(rng, 2000, 12000)
    return _case(waters=waters, **_cube(round((waters * 30.0) ** (1 / 3), 2)), tilt=rng.random() < 0.5, cltype=0,
                 nins=_log(rng, 20, 400), frames=rng.randint(1, 3), flex=flex, host=host, bins=rng.choice([300, 600]))


# ---- inputs ----------------------------------------------------------------


def _cell(case):
    """Cell matrix (columns a, b, c); the skewed one leans b and c by a quarter of a box."""
    m = np.diag([case["lx"], case["ly"], case["lz"]]).astype(np.float64)
    if case["tilt"]:
        m[0, 1], m[1, 2] = 0.25 * case["lx"], -0.25 * case["ly"]
    return m.astype(np.float32)


def _species(case):
    """(solvent species, solute species) of a case: the same for every seed."""
    rng = np.random.default_rng(1000 * case["sites"] + case["chain_sites"])
    solvent = []
    if case["waters"]:
        solvent.append(synth.water_species(case["waters"]))
    if case["chains"]:
        n = case["chain_sites"]
        q = rng.normal(0.0, 0.2, n)
        solvent.append(Species("chain", case["chains"], q - q.mean(), rng.uniform(0.03, 0.2, n), rng.uniform(3.0, 4.0, n),
                               synth.random_chain(rng, n)))
    if case["layout"] == "slab":
        solvent.reverse()
    m = case["solutes"]
    counts = [case["sites"]] if m == 1 else [round(math.exp(math.log(case["sites"]) * k / (m - 1))) for k in range(m)]
    solutes = [synth.tetra_species() if n == 5 else synth.random_solute(rng, "solute%d" % k, n)
               for k, n in enumerate(counts)]
    for s in solutes:
        if s.nsite == 1:
            s.charge[:] = 0.0
    return solvent, solutes


def _positions(case, solvent, solute, rng):
    """One frame's sites, [atoms, 3] float32, in the order of the topology."""
    box = np.array([case["lx"], case["ly"], case["lz"]])
    parts = []
    if case["mode"] == "soln":
        g = solute.geometry + (rng.normal(0.0, 0.1, solute.geometry.shape) if case["flex"] else 0.0)
        g = box / 2 + g @ synth.random_rotations(rng, 1)[0].T
        n = solvent[0].nmol
        wc = synth.lattice_centres(rng, n, box, avoid=g, avoid_r=3.2, spare=max(64, n // 40) + 12 * solute.nsite)
        parts = [g, synth.place_rigid(rng, solvent[0].geometry, wc)]
    elif case["layout"] == "mixed":
        centres = synth.lattice_centres(rng, sum(s.nmol for s in solvent), box)
        at = 0
        for s in solvent:
            parts.append(synth.place_rigid(rng, s.geometry, centres[at:at + s.nmol]))
            at += s.nmol
    else:
        for s in solvent:
            n, chain = s.nmol, s.name == "chain"
            if case["layout"] == "slab" and not chain:
                k = n // 2
                c = np.concatenate([synth.region_lattice(rng, k, (0, 0, 0), (box[0], box[1], 0.3 * box[2])),
                                    synth.region_lattice(rng, n - k, (0, 0, 0.7 * box[2]), box)])
            else:
                z0, z1 = (0.3, 0.7) if case["layout"] == "slab" else (0.15, 0.45) if chain else (0.04, 0.54)
                c = synth.region_lattice(rng, n, (0, 0, z0 * box[2]), (box[0], box[1], z1 * box[2]))
            parts.append(synth.place_rigid(rng, s.geometry, c))
    x = np.concatenate(parts)
    if case["tilt"]:  # the lattice of the upright box, sheared with the cell
        x = (x / box) @ _cell(case).astype(np.float64).T
    return np.ascontiguousarray(x, np.float32)


def _insertions(case, solute, rng):
    box = np.array([case["lx"], case["ly"], case["lz"]])
    z0, z1 = {"mixed": (0.0, 1.0), "slab": (0.3, 0.7), "vapour": (0.7, 0.9)}[case["layout"]]
    n = case["nins"]
    c = rng.uniform(0.0, 1.0, (n, 3)) * np.array([1.0, 1.0, z1 - z0]) + np.array([0.0, 0.0, z0])
    c = c @ _cell(case).astype(np.float64).T if case["tilt"] else c * box
    conf = np.broadcast_to(solute.geometry, (n, solute.nsite, 3))
    if case["flex"]:
        conf = conf + rng.normal(0.0, 0.1, conf.shape)
    x = c[:, None, :] + np.einsum("nij,nsj->nsi", synth.random_rotations(rng, n), conf)
    return np.ascontiguousarray(x, np.float32)


def _inputs(case, seed):
    """Host inputs of a case: ([frame sites], [[insertions of each solute] of each frame])."""
    rng = np.random.default_rng(int(seed) + 1)
    solvent, solutes = _species(case)
    pos = [_positions(case, solvent, solutes[0], rng) for _ in range(case["frames"])]
    ins = [[] if case["mode"] == "soln" else [_insertions(case, s, rng) for s in solutes] for _ in range(case["frames"])]
    return solvent, solutes, pos, ins


def _mesh(case, nspecies):
    """The energy mesh of one species and its open-ended part, repeated for every species."""
    if case["mode"] == "soln":
        mesh, core = synth.linear_log_mesh(-60.0, 60.0, 120.0 / case["bins"], 0, 0)
    else:
        lo = -150.0 if case["chains"] and case["chain_sites"] > 20 else -60.0 if case["chains"] or case["sites"] > 5 else -20.0
        nlog = case["bins"] // 6
        mesh, core = synth.linear_log_mesh(lo, 5.0, (5.0 - lo) / (case["bins"] - nlog), 1.0e4, nlog)
    return (np.full(nspecies, len(mesh), np.int32), np.full(nspecies, len(mesh) - core, np.int32),
            np.tile(np.asarray(mesh, np.float64), nspecies))


def _params(case):
    st = 1 if case["mode"] == "soln" else 3 if case["flex"] else 2
    return hot_path_params(st, (case["ms1"], case["ms2"], case["ms3"]), splodr=case["order"], cltype=case["cltype"],
                           corrcal=int(case["corr"]))


def prepare(case, seed):
    solvent, solutes, pos, ins = _inputs(case, seed)
    soln = case["mode"] == "soln"
    topo = build_topology([solutes[0]] + solvent if soln else solvent + [solutes[0]],
                          solute_index=0 if soln else len(solvent), refs=not soln,
                          extra_lj_species=solutes if len(solutes) > 1 else None)
    ctx = capi.Context(topo, _params(case))
    ctx.set_mesh(*_mesh(case, topo.numslv))
    if soln:
        ctx.set_solute_molecules(topo.tagslt)
    elif len(solutes) == 1:
        ctx.set_solute(topo.slt_ljtype, topo.slt_charge32)
    else:
        tops = [build_topology(solvent + [s], solute_index=len(solvent), refs=True, extra_lj_species=solutes)
                for s in solutes]
        ctx.set_solutes([(t.slt_ljtype, t.slt_charge32) for t in tops])
    if not case["host"]:
        pos = [torch.from_numpy(x).cuda() for x in pos]
        ins = [[torch.from_numpy(x).cuda() for x in per] for per in ins]
        torch.cuda.synchronize()
    st = dict(ctx=ctx, pos=pos, ins=ins, cell=_cell(case), host=case["host"], soln=soln, out=case["out"],
              nslt=len(topo.tagslt), nsolute=len(solutes), graph=None)
    if case["graph"]:
        _frames(st)
        ctx.sync()
        ctx.graph_begin()
        _frames(st)
        st["graph"] = ctx.graph_end()
    return st


def _frames(st):
    """The frames of a block; in solution runs each frame's solvation energies are read, as erdst writes them."""
    ctx, fl = st["ctx"], []
    for x, per in zip(st["pos"], st["ins"]):
        if st["host"]:
            ctx.set_frame(x, st["cell"])
        else:
            ctx.set_frame_device(x.data_ptr(), st["cell"])
        for k, s in enumerate(per):
            if st["nsolute"] > 1:
                ctx.select_solute(k)
            if st["host"]:
                ctx.set_insertions(s)
            else:
                ctx.set_insertions_device(s.shape[0], s.data_ptr())
        ctx.run(capi.ER_BATCHED)
        if st["soln"]:
            ctx.sync()
            fl.append(ctx.flceng(st["nslt"]))
    return fl


def run(st):
    ctx = st["ctx"]
    if st["out"] == "energies":
        _frames(st)
        ctx.sync()
        u, u0 = ctx.uvengy()
        return {"uvengy": u, "uvengy0": u0}
    ctx.clear()
    if st["graph"] is not None:
        ctx.graph_launch(st["graph"])
        fl = []
    else:
        fl = _frames(st)
    ctx.sync()
    got = []
    for k in range(st["nsolute"]):
        if st["nsolute"] > 1:
            ctx.select_solute(k)
        g = ctx.fetch()
        got.append({"edens": g["edens"], "ecorr": g["ecorr"], "minuv": g["minuv"], "maxuv": g["maxuv"],
                    "scal": np.array([g["engnorm"], g["engsmpl"], g["avslf"], g["voffset"]])})
        if st["soln"]:
            got[-1].update(slnuv=g["slnuv"], flceng=fl)
    return got


def work(case):
    """Inputs and results once each; the operations of the physics: site pairs within the cutoff, two
    half-size transforms of each insertion's grid, its gather at every atom, the binning and the correlations."""
    solvent, solutes = _species(case)
    atoms = sum(s.nmol * s.nsite for s in solvent)
    mols = sum(s.nmol for s in solvent)
    ermax = case["bins"] * len(solvent)
    V, G = case["lx"] * case["ly"] * case["lz"], case["ms1"] * case["ms2"] * case["ms3"]
    in_cut = min(atoms, atoms / V * 4.0 / 3.0 * math.pi * 12.0 ** 3)
    per_frame = 1 if case["mode"] == "soln" else case["nins"]
    sites = sum(s.nsite for s in solutes)
    n = per_frame * len(solutes)
    flops = per_frame * sites * in_cut * 40.0 + n * mols * 2.0
    if case["cltype"]:
        flops += n * (2 * 2.5 * G * math.log2(G) + 2.0 * G + atoms * (2.0 * case["order"] ** 3 + 2 * case["order"] ** 2))
    if case["corr"]:
        flops += 1.0 * n * ermax * (ermax + 1)
    size = atoms * 12.0 + per_frame * sites * 12.0
    total = case["frames"] * size + atoms * 8.0
    total += (n * mols + n) * 4.0 if case["out"] == "energies" else \
        len(solutes) * 8.0 * (ermax + (ermax * ermax if case["corr"] else 0))
    return {"bytes": total, "flops": case["frames"] * flops}


# ---- the same results in 64 bits ---------------------------------------------

_QSCALE = 18.22261721


def _spline(t, order):
    """M_order(t + c), c = 0 .. order-1, of fractions t: [..., order]."""
    w = [t, 1.0 - t]
    for k in range(3, order + 1):
        z = torch.zeros_like(t)
        prev = [z] + w + [z]  # prev[c + 1] = M_{k-1}(t + c)
        w = [((t + c) * prev[c + 1] + (k - c - t) * prev[c]) / (k - 1) for c in range(k)]
    return torch.stack(w, -1)


class _Mesh64:
    """The particle-mesh sum of one case in 64 bits on `dev`."""

    def __init__(self, case, cell, screen, dev):
        self.K = K = [case["ms1"], case["ms2"], case["ms3"]]
        self.order = n = case["order"]
        self.inv = torch.linalg.inv(cell)
        vol = float(torch.linalg.det(cell))
        m = [torch.fft.fftfreq(k, 1.0 / k, dtype=torch.float64, device=dev) for k in K]
        # |b(m)|^2 of each axis: the transform of the spline at the grid points
        w = _spline(torch.zeros(1, dtype=torch.float64, device=dev), n)[0]
        b = []
        for d in range(3):
            ph = 2 * math.pi * torch.arange(n, dtype=torch.float64, device=dev)[None, :] * m[d][:, None] / K[d]
            b.append((w[None, :] * torch.cos(ph)).sum(1) ** 2 + (w[None, :] * torch.sin(ph)).sum(1) ** 2)
        m[2], b[2] = m[2][: K[2] // 2 + 1].abs(), b[2][: K[2] // 2 + 1]
        g = torch.stack(torch.meshgrid(*m, indexing="ij"), -1) @ self.inv  # sum_i m_i inv[i, :]
        r2 = (g * g).sum(-1)
        f = torch.exp(-math.pi ** 2 * r2 / screen ** 2) / r2 / math.pi / vol
        f = f / (b[0][:, None, None] * b[1][None, :, None] * b[2][None, None, :])
        f[0, 0, 0] = 0.0
        if n % 2:
            for d in range(3):
                if K[d] % 2 == 0:
                    f.select(d, K[d] // 2).zero_()
        self.f = f

    def stencil(self, x):
        """(flat grid indices, weights) of sites x: [sites, order^3] each."""
        s = x @ self.inv.T
        s = s - torch.floor(s)
        idx, wts = [], []
        for d, k in enumerate(self.K):
            u = s[:, d] * k
            g = torch.floor(u).to(torch.int64)
            wts.append(_spline(u - g, self.order))
            idx.append((g[:, None] - torch.arange(self.order, device=x.device)) % k)
        at = ((idx[0][:, :, None, None] * self.K[1] + idx[1][:, None, :, None]) * self.K[2] + idx[2][:, None, None, :])
        w = wts[0][:, :, None, None] * wts[1][:, None, :, None] * wts[2][:, None, None, :]
        return at.reshape(len(x), -1), w.reshape(len(x), -1)

    def potential(self, x, q):
        """(the grid potential of charges q at x, their reciprocal self energy)."""
        at, w = self.stencil(x)
        rho = torch.zeros(self.K[0] * self.K[1] * self.K[2], dtype=torch.float64, device=x.device)
        rho.index_add_(0, at.reshape(-1), (q[:, None] * w).reshape(-1))
        phi = torch.fft.irfftn(torch.fft.rfftn(rho.view(self.K)) * self.f, self.K, norm="forward").reshape(-1)
        return phi, 0.5 * (rho * phi).sum()


def exact(case, seed):
    dev = torch.device("cuda" if torch.cuda.is_available() else "cpu")
    f64 = lambda v: torch.as_tensor(np.asarray(v, np.float64), device=dev)  # noqa: E731
    solvent, solutes, pos, ins = _inputs(case, seed)
    prm = _params(case)
    soln, bare = case["mode"] == "soln", case["cltype"] == 0
    # the parameters as the library receives them: 32-bit values
    cut, up, lw, screen = (float(np.float32(prm[k])) for k in ("elecut", "upljcut", "lwljcut", "screen"))
    kT, order_q = prm["temp"], np.float32(_QSCALE)
    cell = f64(_cell(case))
    vol, inv = float(torch.linalg.det(cell)), torch.linalg.inv(cell)
    per_site = lambda v: np.concatenate([np.tile(np.asarray(v(s), np.float32), s.nmol) for s in solvent])  # noqa: E731
    q = f64(np.float32(order_q * per_site(lambda s: s.charge)))
    eps32, sig32 = per_site(lambda s: s.eps), per_site(lambda s: s.sigma)
    sites = np.concatenate([np.full(s.nmol, s.nsite) for s in solvent])
    mol = torch.as_tensor(np.repeat(np.arange(len(sites)), sites), device=dev)
    nmol = len(sites)
    molq = torch.zeros(nmol, dtype=torch.float64, device=dev).index_add_(0, mol, q)
    species = np.repeat(np.arange(len(solvent)), [s.nmol for s in solvent])
    uvmax, _, uvcrd = _mesh(case, len(solvent))
    bins, ermax = int(uvmax[0]), int(uvmax.sum())
    edges = f64(uvcrd[:bins])
    sp_off = torch.as_tensor(species * bins, device=dev)
    mesh = None if bare else _Mesh64(case, cell, screen, dev)

    def image(d):
        f = torch.round(d[..., 2] / cell[2, 2])
        d = d - f[..., None] * cell[:, 2]
        f = torch.round(d[..., 1] / cell[1, 1])
        d = d - f[..., None] * cell[:, 1]
        f = torch.round(d[..., 0] / cell[0, 0])
        return d - f[..., None] * cell[:, 0]

    def pairs(x, qs, le, ls, xs):
        """Per-molecule real-space energy of solute sites x against the solvent sites xs."""
        out = torch.zeros(nmol, dtype=torch.float64, device=dev)
        step = max(1, 20_000_000 // len(xs))
        for s0 in range(0, len(x), step):
            d = image(x[s0:s0 + step, None, :] - xs[None, :, :])
            r2 = (d * d).sum(-1)
            s, a = torch.nonzero(r2 < max(cut, up) ** 2, as_tuple=True)
            r2 = r2[s, a]
            r, s = torch.sqrt(r2), s + s0
            i6 = (ls[s, a] / r2) ** 3
            lj = 4.0 * le[s, a] * i6 * (i6 - 1.0)
            sw = (2 * r2 + up ** 2 - 3 * lw ** 2) * (r2 - up ** 2) ** 2 / (up ** 2 - lw ** 2) ** 3
            lj = torch.where(r > up, torch.zeros_like(lj), torch.where(r > lw, sw * lj, lj))
            cl = qs[s] * q[a] / r
            if not bare:
                cl = cl * torch.special.erfc(screen * r)
            out.index_add_(0, mol[a], lj + torch.where(r >= cut, torch.zeros_like(cl), cl))
        return out

    got = []
    for k, slt in enumerate(solutes):
        e32, s32 = np.asarray(slt.eps, np.float32)[:, None], np.asarray(slt.sigma, np.float32)[:, None]
        le, ls = f64(np.sqrt(e32 * eps32)), f64(((s32 + sig32) / np.float32(2.0)) ** 2)
        qs = f64(np.float32(order_q * np.asarray(slt.charge, np.float32)))
        Q = float(qs.sum())
        ns = slt.nsite
        us, u0s, per_frame = [], [], 1 if soln else case["nins"]
        first_real = None
        for f in range(case["frames"]):
            xs = f64(pos[f][ns:] if soln else pos[f])
            xi = f64(pos[f][None, :ns] if soln else ins[f][k])
            at, w = (None, None) if bare else mesh.stencil(xs)
            for n in range(per_frame):
                u = pairs(xi[n], qs, le, ls, xs)
                u0 = 0.0
                if not bare:
                    phi, rec = mesh.potential(xi[n], qs)
                    u.index_add_(0, mol, q * (w * phi[at]).sum(1))
                    u -= math.pi * Q * molq / screen ** 2 / vol
                    d = image(xi[n][:, None, :] - xi[n][None, :, :])
                    r = torch.sqrt((d * d).sum(-1))
                    i, j = torch.triu_indices(ns, ns, 1, device=dev)
                    real = -(qs * qs).sum() * screen / math.sqrt(math.pi) \
                        - (qs[i] * qs[j] * torch.special.erf(screen * r[i, j]) / r[i, j]).sum()
                    if first_real is None:
                        first_real = real
                    if not soln and not case["flex"]:
                        real = first_real
                    u0 = float(rec + real) - 0.5 * math.pi * Q * Q / screen ** 2 / vol
                us.append(u)
                u0s.append(u0)
        if case["out"] == "energies":
            return {"uvengy": torch.stack(us).cpu().numpy(), "uvengy0": np.array(u0s)}
        U, u0 = torch.stack(us), f64(u0s)
        wgt = torch.full_like(u0, vol)
        if not bare:
            qtot = float(molq.sum()) + (Q if soln else 0.0)
            wgt = wgt * math.exp(math.pi * qtot ** 2 / screen ** 2 / vol / 2.0 / kT)
        avslf, voff = float(wgt.sum()), 0.0
        if prm["wgtslf"]:
            voff = u0s[0]
            wgt = wgt * torch.exp(-(u0 - voff) / kT)
        b = torch.clamp(torch.searchsorted(edges, U.contiguous()), min=1) - 1 + sp_off[None, :]
        C = torch.zeros(len(U), ermax, dtype=torch.float64, device=dev)
        C.scatter_add_(1, b, torch.ones_like(U))
        ecorr = (C * wgt[:, None]).T @ C if case["corr"] else torch.zeros(ermax, ermax, dtype=torch.float64, device=dev)
        lo, hi = [float(u0.min())], [float(u0.max())]
        fl = []
        for s in range(len(solvent)):
            cols = U[:, torch.as_tensor(species == s, device=dev)]
            lo.append(float(cols.min()))
            hi.append(float(cols.max()))
            fl.append(cols.sum(1))
        fl = torch.stack(fl, 1)
        one = {"edens": (C * wgt[:, None]).sum(0).cpu().numpy(), "ecorr": ecorr.cpu().numpy(),
               "minuv": np.array(lo), "maxuv": np.array(hi), "scal": np.array([float(wgt.sum()), len(U), avslf, voff])}
        if soln:
            one.update(slnuv=(fl * wgt[:, None]).sum(0).cpu().numpy(), flceng=[v[None].cpu().numpy() for v in fl])
        got.append(one)
    return got
