"""The work that is measured: calls of the framework's public entry points over the sizes a user runs.

A case is a dict of plain values; `prepare` builds what a program holds before
the call, `run` makes one pass, `work` says what the pass cannot do without and
`exact` gives its results in 64 bits from plain torch / numpy.  The systems are
the seeded spheres of `q6_amd.synth` (the benchmark's 30 A sphere of 400
ten-atom solute groups and TIP3P, the 20 A water sphere around one 12-atom
chain, the uneven spheres, the 18 A sphere of a nine-site solvent), relaxed here
with a plain soft-sphere descent so that every evaluation and every run starts
from a structure without overlaps.  The topology of a case is the same for
every seed; positions, velocities, frames and energies come from the seed.

Results of the mixed path are FP32 pair arithmetic: the program keeps them in
single precision, as Q's trajectory files (write_trj) hold coordinates.
"""
import functools
import math

import numpy as np
import torch

from q6_amd import abi, adjoint, synth
from q6_amd.engine import NonbondedEngine
from q6_amd.md import BatchMD, free_energy

ENERGIES = ("pp_el", "pp_vdw", "pw_el", "pw_vdw", "ww_el", "ww_vdw", "lrf", "solvent_radial", "water_pol")
Q_ENERGIES = ("qq_el", "qq_vdw", "qp_el", "qp_vdw", "qw_el", "qw_vdw")
PRECISION = {"fp64": abi.QNB_PREC_FP64, "mixed": abi.QNB_PREC_MIXED}


def listed():
    bench = dict(radius=30.0, chains=400, beads=10, qchains=3, states=2)
    water = dict(radius=20.0, chains=1, beads=12, qchains=1, states=2)
    return [
        # lambda-window FEP: the benchmark's 51 windows in one batch, five list cycles between two saved structures
        dict(name="md_windows51", kind="md", precision="mixed", windows=51, steps=50, **bench),
        # independent systems of different size in one batch (four spheres of 15 to 27 A, 2 and 3 states)
        dict(name="md_uneven", kind="md", precision="mixed", windows=4, steps=40, radius=15.0, grow=4.0, chains=42,
             beads=10, qchains=2, states=3),
        # one window on the plain FP64 path: equilibration, and the reference a user checks the mixed path with
        dict(name="md_single_fp64", kind="md", precision="fp64", windows=1, steps=40, **bench),
        # the smallest run: one molecule in a water sphere, where launches and latency count
        dict(name="md_small", kind="md", precision="mixed", windows=1, steps=40, **water),
        # Qdyn6's own loop calling the engine every step with host arrays: every term of one step, FP64
        dict(name="eval_fp64", kind="eval", precision="fp64", **bench),
        # the same call in mixed precision on ragged sizes: 7-atom groups, Q-atoms bonded to other atoms, 3 states
        dict(name="eval_mixed_ragged", kind="eval", precision="mixed", radius=23.0, chains=101, beads=7, qchains=3,
             states=3, qper=5),
        # every tenth step of that loop: pair lists and LRF expansion of a large, water-rich sphere
        dict(name="lists_large", kind="lists", precision="fp64", radius=36.0, chains=24, beads=11, qchains=2, states=2),
        # a flexible nine-site solvent instead of water (single evaluations only)
        dict(name="eval_solvent9", kind="solvent9", precision="fp64", radius=18.0, chains=6, beads=10, qchains=1,
             states=2),
        # EVB calibration: parameter derivatives over the frames that a batch keeps on the device
        dict(name="adjoint_batch", kind="adjoint_batch", precision="mixed", windows=6, frames=20, radius=24.0,
             chains=120, beads=10, qchains=3, states=2),
        # the same for frames a program read from trajectory files
        dict(name="adjoint_frames", kind="adjoint", precision="fp64", frames=24, radius=18.0, chains=20, beads=9,
             qchains=2, states=3),
        # Qfep6's analysis of a whole run: 51 windows, reaction free energy along the gap
        dict(name="free_energy", kind="fep", windows=51, frames=1000, bins=50),
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(("md", "md", "md", "eval", "eval", "lists", "solvent9", "adjoint_batch", "adjoint", "fep"))
    if kind == "fep":
        return dict(kind=kind, windows=rng.randint(5, 61), frames=int(_log(rng, 50, 1500)), bins=rng.randint(10, 60))
    radius = round(_log(rng, 13.0, 20.0 if kind == "solvent9" else 29.0), 2)
    beads = rng.randint(5, 13)
    # solute from one molecule to a third of the sphere's atoms
    chains = max(2, int(_log(rng, 2.0, 0.13 * radius ** 3 / beads)))
    if kind == "solvent9":
        chains = min(chains, 8)
    qchains = rng.randint(1, min(3, chains))
    case = dict(kind=kind, precision=rng.choice(("mixed", "mixed", "fp64")), radius=radius, chains=chains, beads=beads,
                qchains=qchains, states=rng.randint(1, 4) if kind in ("md", "eval", "lists") else rng.randint(2, 3))
    if rng.random() < 0.5:
        case["qper"] = rng.randint(3, beads)
    if kind == "md":
        # at most the atoms that the 51 windows of the 30 A sphere hold
        case["windows"] = max(1, min(51, int(_log(rng, 1.0, 51.0)), int(550000 / (0.42 * radius ** 3))))
        case["steps"] = 10 * rng.randint(2, 4)
        if rng.random() < 0.3 and case["windows"] <= 6:
            case["grow"] = round(rng.uniform(0.5, 1.5), 2)
            case["windows"] = max(2, case["windows"])
    elif kind in ("adjoint", "adjoint_batch"):
        case["frames"] = rng.randint(5, 24)
        case["radius"] = min(radius, 22.0)
        case["chains"] = min(chains, 60)
        if kind == "adjoint_batch":
            case["windows"] = rng.randint(1, 8)
    return case


# ------------------------------------------------------------- systems

def _soft_spheres(x, nsol, nbead, nsolvent, sa, iters=250):
    """Moves beads and whole solvent molecules apart until heavy sites are near
    contact distance (2.9 A); bonds and the 1-3 distances of the chains are
    pulled back to their lengths.  Plain torch, sums in a fixed order."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    x = torch.tensor(x, dtype=torch.float64, device=dev)
    nchain = nsol // nbead
    first = nsol + sa * torch.arange(nsolvent, device=dev)
    ids = torch.cat([torch.arange(nsol, device=dev), first])
    chain = torch.where(ids < nsol, ids // nbead, -1 - ids)
    p = x[ids].float()
    for _ in range(iters):
        move = torch.zeros_like(p)
        for lo in range(0, len(p), 4096):
            u = p[lo:lo + 4096, None, :] - p[None, :, :]
            r = u.square().sum(-1).sqrt()
            near = (chain[lo:lo + 4096, None] == chain[None, :]) & ((ids[lo:lo + 4096, None] - ids[None, :]).abs() <= 2)
            w = torch.where(near | (r < 1e-3), torch.zeros_like(r), (2.9 - r).clamp_min(0.0) / r.clamp_min(1e-3))
            move[lo:lo + 4096] = 0.25 * (u * w[..., None]).sum(1)
        if nchain:
            c = p[:nsol].view(nchain, nbead, 3)
            m = move[:nsol].view(nchain, nbead, 3)
            for step, length in ((1, 1.5), (2, 2.45)):
                if nbead > step:
                    u = c[:, step:] - c[:, :-step]
                    r = u.square().sum(-1, keepdim=True).sqrt()
                    g = 0.25 * (r - length) / r * u
                    m[:, :-step] += g
                    m[:, step:] -= g
        size = move.square().sum(-1, keepdim=True).sqrt()
        p = p + move * (0.2 / size.clamp_min(0.2))
    move = (p - x[ids].float()).double()
    x[:nsol] += move[:nsol]
    if nsolvent:
        x[nsol:] = (x[nsol:].view(nsolvent, sa, 3) + move[nsol:, None, :]).view(-1, 3)
    return x.cpu().numpy()


@functools.lru_cache(maxsize=None)
def _sphere(radius, chains, beads, qchains, states, qper, nine):
    """A relaxed sphere; the same system for the same sizes."""
    lam = np.arange(states, 0, -1) / (states * (states + 1) / 2)
    if nine:
        s = synth.build(radius, chains, beads, qchains, states, 41, chain_region=0.35 * radius, q_sigma=0.4,
                        lambdas=lam, compact=3.0, q_per_chain=qper, water_fill=radius - 1.0, **synth.PACK)
        s = synth.replace_solvent(s, synth.ethanol(), 0.0085, 48)
    else:
        s = synth.build(radius, chains, beads, qchains, states, 11, chain_region=0.55 * radius, q_sigma=0.3,
                        lambdas=lam, compact=3.0, q_per_chain=qper, water_fill=radius, **synth.PACK)
    s.x = np.ascontiguousarray(_soft_spheres(s.x, s.n["nat_solute"], beads, s.n["nwat"], s.n["solv_atom"]))
    return s


def _system(case, k=0):
    f = case.get("grow", 0.0) * k
    scale = (case["radius"] + f) ** 3 / case["radius"] ** 3
    return _sphere(case["radius"] + f, max(case["qchains"], int(case["chains"] * scale)), case["beads"],
                   case["qchains"], case["states"] if f == 0.0 or case["states"] < 3 else 2 + k % 2,
                   case.get("qper"), case["kind"] == "solvent9")


def _moved(s, rng):
    """A thermal copy of the positions: every solute atom and every whole
    solvent molecule displaced."""
    nsol, nw, sa = s.n["nat_solute"], s.n["nwat"], s.n["solv_atom"]
    x = s.x.copy()
    x[:nsol] += rng.normal(0.0, 0.03, (nsol, 3))
    x[nsol:] += np.repeat(rng.normal(0.0, 0.05, (nw, 3)), sa, axis=0)
    return x


def _series(case, seed):
    rng = np.random.default_rng(seed)
    lam1 = np.linspace(1.0, 0.0, case["windows"])
    lam = np.stack([lam1, 1.0 - lam1], 1)
    V = []
    for l1 in lam1:
        gap = rng.normal(-150.0 + 300.0 * l1, 12.0, case["frames"])
        mean = rng.normal(-40.0, 6.0, case["frames"])
        V.append(np.stack([mean - 0.5 * gap, mean + 0.5 * gap], 1))
    r = [rng.uniform(2.0, 4.5, case["frames"]) for _ in lam1]
    par = dict(kT=0.596, nskip=case["frames"] // 20, nbins=case["bins"], nmin=5, alpha=np.array([0.0, 3.5]),
               coeff=np.array([1.0, -1.0]), A=35.0, mu=0.6, eta=0.05, r0=2.0)
    return V, lam, r, par


# ------------------------------------------------------------- the calls

def prepare(case, seed):
    kind = case["kind"]
    if kind == "fep":
        V, lam, r, par = _series(case, seed)
        return dict(case=case, V=V, lam=lam, r=r, par=par)
    rng = np.random.default_rng(seed)
    precision = PRECISION[case["precision"]]
    state = dict(case=case, single=case["precision"] == "mixed")
    if kind in ("md", "adjoint_batch"):
        n = case["windows"]
        systems = [_system(case, k) for k in range(n)] if "grow" in case else [_system(case)] * n
        lambdas = []
        for k, s in enumerate(systems):
            lam = np.asarray(s.par["lambda"], float)
            t = k / max(n - 1, 1)
            lambdas.append((1.0 - t) * lam + t * lam[::-1])
        steps = case["steps"] if kind == "md" else case["frames"]
        # the history holds one pass's sampled energies
        b = BatchMD(systems, lambdas, [synth.maxwell_velocities(s, 300.0, seed + 7 * k) for k, s in enumerate(systems)],
                    precision=precision, nbcycle=10, ene_every=10, max_frames=max(1, steps // 10), tau_T_fs=20.0,
                    positions=[_moved(s, rng) for s in systems])
        state.update(batch=b, systems=systems)
        if kind == "md":
            b.prepare_graph()
        else:
            b.store_frames(1, case["frames"])
            b.run(steps)
            b.sync()
            made = {id(s): adjoint.tangent_struct(s) for s in systems}
            state.update(made=made, tangents=[made[id(s)][0] for s in systems])
        return state
    s = _system(case)
    engine = NonbondedEngine(s, precision=precision)
    x = _moved(s, rng)
    state.update(engine=engine, system=s, x=x)
    if kind in ("eval", "solvent9"):
        engine.make_pair_lists(x)
    elif kind == "adjoint":
        tangent, keep = adjoint.tangent_struct(s)
        state.update(tangent=tangent, keep=keep, frames=np.stack([_moved(s, rng) for _ in range(case["frames"])]))
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "fep":
        r = free_energy(state["V"], state["lam"], rkl=state["r"], **state["par"])
        return {k: r[k] for k in ("dgf", "dgr", "dG", "gap_range", "dGg", "c1", "npts", "binned", "binned_c1",
                                  "binned_r", "ptsum")}
    kept = np.float32 if state["single"] else np.float64
    if kind == "md":
        b = state["batch"]
        b.run(case["steps"])
        b.sync()
        out = {}
        for k in range(b.n):
            x, v = b.state(k)
            out["x%d" % k] = x.astype(kept)
            if not state["single"]:  # a restart file holds the FP64 run's velocities too
                out["v%d" % k] = v
        out["energies"] = np.stack([b.energies(k) for k in range(b.n)]).astype(kept)
        return out
    if kind == "adjoint_batch":
        return [a.astype(kept) for a in state["batch"].adjoint(state["tangents"])]
    engine = state["engine"]
    if kind in ("eval", "solvent9"):
        d, E, EQ = engine.eval_terms(abi.T_ALL, state["x"], Tfree=300.0)
        return {"d": d.astype(kept), "E": np.array([E[k] for k in ENERGIES], kept),
                "EQ": np.array([[q[k] for k in Q_ENERGIES] for q in EQ], kept)}
    if kind == "lists":
        engine.make_pair_lists(state["x"])
        return engine.lrf().astype(kept)
    return engine.adjoint(state["tangent"], state["frames"]).astype(kept)


def work(case):
    """Pairs and LRF updates from the mean densities (0.1 atoms and one charge
    group per 40 A^3), positions, gradients and tables moved once."""
    kind = case["kind"]
    if kind == "fep":
        n = case["windows"] * case["frames"]
        return {"bytes": 24.0 * n, "flops": 120.0 * n}

    def atoms(k):
        return 0.42 * (case["radius"] + case.get("grow", 0.0) * k) ** 3

    nst, nq = case["states"], case["qchains"] * case.get("qper", case["beads"])
    nat = [atoms(k) for k in range(case.get("windows", 1))]
    sweep = sum(89.0 * a * a / 4.0 for a in nat)
    pairs = sum(a * (28.0 * 180 + nq * (12 + 20.0 * nst)) for a in nat)
    if kind == "md":
        return {"bytes": case["steps"] * sum(nat) * 104.0, "flops": case["steps"] * (pairs + sweep / 10.0)}
    if kind == "lists":
        return {"bytes": nat[0] * (24 + 86.0), "flops": sweep}
    if kind in ("adjoint", "adjoint_batch"):
        return {"bytes": case["frames"] * sum(nat) * 24.0, "flops": case["frames"] * sum(nat) * nq * (10 + 15.0 * nst)}
    return {"bytes": nat[0] * 48.0, "flops": pairs}


# ------------------------------------------------------------- in 64 bits

def exact(case, seed):
    kind = case["kind"]
    if kind == "fep":
        return _exact_fep(case, seed)
    if kind in ("md", "adjoint_batch"):  # whole runs: no value of their own beyond a few steps
        return None
    s = _system(case)
    rng = np.random.default_rng(seed)
    x = _moved(s, rng)
    if kind in ("eval", "solvent9"):
        return _exact_terms(s, x)
    if kind == "lists":
        return _lrf_table(s, _t(x)).cpu().numpy()
    return _exact_adjoint(s, [_moved(s, rng) for _ in range(case["frames"])])


def _t(a):
    return torch.as_tensor(np.asarray(a), dtype=torch.float64, device="cuda" if torch.cuda.is_available() else "cpu")


def _ti(a):
    return torch.as_tensor(np.asarray(a, np.int64), device="cuda" if torch.cuda.is_available() else "cpu")


def _reference_atoms(s):
    n = s.n
    return _ti(np.concatenate([s.a["cgp_iswitch"][:n["ncgp_solute"]], n["nat_solute"] + n["solv_atom"] * np.arange(n["nwat"])]))


def _group_of(s):
    g = np.zeros(s.natom, np.int64)
    for k in range(s.n["ncgp"]):
        g[s.a["cgpatom"][s.a["cgp_first"][k]:s.a["cgp_last"][k] + 1]] = k
    return _ti(g)


def _inside(s, p):
    """Group pairs within the class cut-off: |p_a - p_b|^2 between reference atoms."""
    r2 = (p[:, None, :] - p[None, :, :]).square().sum(-1)
    sol = torch.arange(len(p), device=p.device) < s.n["ncgp_solute"]
    cut = torch.where(sol[:, None] & sol[None, :], s.par["Rcpp"] ** 2,
                      torch.where(sol[:, None] | sol[None, :], s.par["Rcpw"] ** 2, s.par["Rcww"] ** 2))
    eye = torch.eye(len(p), dtype=torch.bool, device=p.device)
    return (r2 <= cut) & ~eye, (r2 > cut) & (r2 <= s.par["RcLRF"] ** 2) & ~eye


def _lrf_table(s, x):
    """Third-order expansion of the far groups' potential about every group's centre."""
    far = _inside(s, x[_reference_atoms(s)])[1]
    g = _group_of(s)
    n = s.n["ncgp"]
    onehot = torch.zeros(n, s.natom, dtype=torch.float64, device=x.device)
    onehot[g, torch.arange(s.natom, device=x.device)] = 1.0
    centre = onehot @ x / onehot.sum(1, keepdim=True)
    q = _t(s.a["crg"]) * (_ti(s.a["iqatom"]) == 0)
    out = torch.zeros(n, 43, dtype=torch.float64, device=x.device)
    eye = torch.eye(3, dtype=torch.float64, device=x.device)
    for lo in range(0, n, 128):
        hi = min(n, lo + 128)
        c = centre[lo:hi]
        d = x[None, :, :] - c[:, None, :]
        r2 = d.square().sum(-1)
        w = torch.where(far[lo:hi][:, g], q[None, :], torch.zeros_like(r2))
        r = r2.sqrt().clamp_min(1e-9)
        f0, f1 = w / r ** 3, 3.0 * w / r ** 5
        f5 = -15.0 * w / r ** 7
        h = (f1[..., None] * d).sum(1)
        p2 = torch.einsum("aj,ajk->ak", f1, (d[..., :, None] * d[..., None, :]).flatten(2)).view(-1, 3, 3)
        p3 = torch.stack([torch.stack([((f5 * d[..., i] * d[..., j])[..., None] * d).sum(1) for j in range(3)], 1)
                          for i in range(3)], 1)
        p3 = p3 + (torch.einsum("ij,ak->aijk", eye, h) + torch.einsum("ik,aj->aijk", eye, h)
                   + torch.einsum("jk,ai->aijk", eye, h))
        out[lo:hi] = torch.cat([c, (w / r).sum(1, keepdim=True), -(f0[..., None] * d).sum(1),
                                (p2 - eye * f0.sum(1)[:, None, None]).flatten(1), p3.flatten(1)], 1)
    return out


def _lj_coulomb(u, A, B, q):
    """Energies (Coulomb, LJ) and -dE/dr / r of pairs at u."""
    i2 = 1.0 / u.square().sum(-1)
    i1, i6 = i2.sqrt(), i2 ** 3
    el, a, b = q * i1, A * i6 * i6, B * i6
    return el, a - b, i2 * (el + 12.0 * a - 6.0 * b)


def _excluded(s):
    """(i, j) of excluded and of 1-4 solute pairs, each in both orders."""
    out = []
    for win, lst, n in (("listex", "listexlong", "nexlong"), ("list14", "list14long", "n14long")):
        w = np.asarray(s.a[win])[:25 * s.n["nat_solute"]].reshape(-1, 25)
        i, k = np.nonzero(w)
        e = np.stack([i, i + k + 1], 1)
        if s.n.get(n, 0):
            e = np.concatenate([e, np.asarray(s.a[lst]).reshape(-1, 2)])
        out.append(_ti(np.concatenate([e, e[:, ::-1]]) if len(e) else np.zeros((0, 2))))
    return out


def _exact_terms(s, x):
    n, a, par = s.n, s.a, s.par
    nat, nsol, sa, nq, ns = n["natom"], n["nat_solute"], n["solv_atom"], n["nqat"], n["nstates"]
    x = _t(x)
    dev = x.device
    E = dict.fromkeys(ENERGIES, 0.0)
    EQ = torch.zeros(ns, 6, dtype=torch.float64, device=dev)
    d = torch.zeros_like(x)
    g = _group_of(s)
    inside = _inside(s, x[_reference_atoms(s)])[0]
    isq = _ti(a["iqatom"]) > 0
    crg = _t(a["crg"])
    lj = [_t(a[k]).view(-1, 3)[_ti(a["iac"])] for k in ("avdw", "bvdw")]
    site = (torch.arange(nat, device=dev) - nsol) % sa
    table = {k: (_t(a["pw_" + k])[:nsol * sa].view(sa, -1), _t(a["ww_" + k]).view(sa, sa)) for k in ("A", "B", "el")}
    excluded, far14 = _excluded(s)
    for lo in range(0, nat, 1024):
        hi = min(nat, lo + 1024)
        i = torch.arange(lo, hi, device=dev)
        on = inside[g[i]][:, g] | ((g[i][:, None] == g[None, :]) & (i[:, None] < nsol))
        on &= ~isq[i][:, None] & ~isq[None, :] & (i[:, None] != torch.arange(nat, device=dev)[None, :])
        A, B, q = lj[0][i, 0][:, None] * lj[0][None, :, 0], lj[1][i, 0][:, None] * lj[1][None, :, 0], crg[i][:, None] * crg
        w = i >= nsol
        if bool(w.any()):  # solvent rows: the pair tables as the topology gives them
            for M, k in ((A, "A"), (B, "B"), (q, "el")):
                M[w, :nsol] = table[k][0][site[i[w]]]
                M[w, nsol:] = table[k][1][site[nsol:][None, :], site[i[w]][:, None]]
        if bool((~w).any()):
            for M, k in ((A, "A"), (B, "B"), (q, "el")):
                M[~w, nsol:] = table[k][0][site[nsol:]][:, i[~w]].T
        e = excluded[(excluded[:, 0] >= lo) & (excluded[:, 0] < hi)]
        on[e[:, 0] - lo, e[:, 1]] = False
        e = far14[(far14[:, 0] >= lo) & (far14[:, 0] < hi)]
        A[e[:, 0] - lo, e[:, 1]] = lj[0][e[:, 0], 2] * lj[0][e[:, 1], 2]
        B[e[:, 0] - lo, e[:, 1]] = lj[1][e[:, 0], 2] * lj[1][e[:, 1], 2]
        q[e[:, 0] - lo, e[:, 1]] *= s.el14_scale
        r, c = on.nonzero(as_tuple=True)
        u = x[c] - x[lo + r]
        el, vdw, f = _lj_coulomb(u, A[r, c], B[r, c], q[r, c])
        d[lo:hi] += torch.zeros(hi - lo, 3, dtype=torch.float64, device=dev).index_add_(0, r, u * f[:, None])
        kind = (lo + r >= nsol).long() + (c >= nsol).long()
        for k, name in enumerate(("pp", "pw", "ww")):
            E[name + "_el"] = E[name + "_el"] + 0.5 * el[kind == k].sum()
            E[name + "_vdw"] = E[name + "_vdw"] + 0.5 * vdw[kind == k].sum()
    # Q-atoms: with the solvent and the solute within Rcq, bonded neighbours and one another
    iqs, lam = _ti(a["iqseq"])[:nq], _t(par["lambda"])
    qp = {k: _t(a["qp_" + k])[:nsol * nq * ns].view(ns, nq, nsol) for k in ("A", "B", "el", "sc", "set")}
    qw = {k: _t(a["qw_" + k])[:nq * sa * ns].view(ns, sa, nq) for k in ("A", "B", "el", "sc")}
    qq = {k: _t(a["qq_" + k])[:nq * nq * ns].view(ns, nq, nq) for k in ("A", "B", "el", "sc", "set")}
    con = _t(a["qconn3"])[:nsol] != 0
    rc2 = par["Rcq"] ** 2
    ref = x[_reference_atoms(s)].square().sum(-1) <= rc2  # the Q-list centre is the origin
    sol, wat = torch.arange(nsol, device=dev), torch.arange(nsol, nat, device=dev)

    def pair(i, j, A, B, q, sc, st, at):
        u = x[j] - x[i]
        i2 = 1.0 / u.square().sum(-1)
        i6 = 1.0 / (1.0 / i2 ** 3 + sc)
        el, va, vb = q * i2.sqrt(), A * i6 * i6, B * i6
        f = i2 * (el + (12.0 * va - 6.0 * vb) * i6 / i2 ** 3) * lam[st]
        d.index_add_(0, i.reshape(-1), (u * f[..., None]).reshape(-1, 3))
        d.index_add_(0, j.reshape(-1), -(u * f[..., None]).reshape(-1, 3))
        EQ[st, at] += el.sum()
        EQ[st, at + 1] += (va - vb).sum()

    for st in range(ns):
        j = sol[~con & ref[g[sol]]]
        pair(*torch.broadcast_tensors(iqs[:, None], j[None, :]), *(qp[k][st][:, j] for k in ("A", "B", "el", "sc")), st, 2)
        j = wat[ref[g[wat]]]
        pair(*torch.broadcast_tensors(iqs[:, None], j[None, :]),
             *(qw[k][st][site[j]].T for k in ("A", "B", "el", "sc")), st, 4)
        k1, j = ((qp["set"][st] != 0) & (con & ~isq[:nsol])[None, :]).nonzero(as_tuple=True)
        pair(iqs[k1], j, *(qp[k][st][k1, j] for k in ("A", "B", "el", "sc")), st, 2)
        k2, k1 = (qq["set"][st] != 0).nonzero(as_tuple=True)
        pair(iqs[k1], iqs[k2], *(qq[k][st][k2, k1] for k in ("A", "B", "el", "sc")), st, 0)
    # LRF potential of every atom that is not a Q-atom
    L = _lrf_table(s, x)[g]
    dr = L[:, :3] - x
    p1, p2, p3 = L[:, 4:7], L[:, 7:16].view(-1, 3, 3), L[:, 16:].view(-1, 3, 3, 3)
    t2 = torch.einsum("nij,nj->ni", p2, dr)
    q = crg * ~isq
    E["lrf"] = (0.5 * q * (L[:, 3] + (dr * p1).sum(1) + 0.5 * (dr * t2).sum(1))).sum()
    d -= q[:, None] * (p1 + t2 + 0.5 * torch.einsum("nijk,nj,nk->ni", p3, dr, dr))
    # pairs inside every flexible solvent molecule
    inner = n.get("n_solv_int", 0)
    for (i, j), (A, B, q) in zip(np.asarray(a["solv_int_ij"])[:2 * inner].reshape(-1, 2),
                                 np.asarray(a["solv_int_par"])[:3 * inner].reshape(-1, 3)):
        u = x[nsol + int(j)::sa] - x[nsol + int(i)::sa]
        el, vdw, f = _lj_coulomb(u, A, B, q)
        d[nsol + int(i)::sa] += u * f[:, None]
        d[nsol + int(j)::sa] -= u * f[:, None]
        E["ww_el"] = E["ww_el"] + el.sum()
        E["ww_vdw"] = E["ww_vdw"] + vdw.sum()
    _restraints(s, x, d, E)
    return {"d": d.cpu().numpy(), "E": np.array([float(E[k]) for k in ENERGIES]), "EQ": EQ.cpu().numpy()}


def _restraints(s, x, d, E, tfree=300.0):
    """Solvent-sphere surface: radial force and (3-site water) polarisation."""
    n, par = s.n, s.par
    nsol, sa = n["nat_solute"], n["solv_atom"]
    heavy = np.asarray(s.a["heavy"])[nsol:nsol + sa] if sa != 3 else np.array([1, 0, 0])
    v = x[nsol::sa]
    b = v.square().sum(1).sqrt()
    db = b - (par["rwat"] - math.sqrt(par["Boltz"] * tfree / par["fk_wsphere"]))
    e = torch.exp(par["awmz"] * db)
    out = db > 0.0
    erst = torch.where(out, 0.5 * par["fk_wsphere"] * db * db - par["Dwmz"], par["Dwmz"] * (e * e - 2.0 * e))
    dv = torch.where(out, par["fk_wsphere"] * db, -2.0 * par["Dwmz"] * par["awmz"] * (e - e * e)) / b
    for k in np.nonzero(heavy)[0]:
        # the term acts on the heavy atom along its own radial vector of the molecule's first atom
        d[nsol + int(k)::sa] += v * dv[:, None]
        E["solvent_radial"] = E["solvent_radial"] + erst.sum()
    nsh = int(par["nwpolr_shell"])
    if not par["wpol_restr"] or nsh == 0 or sa != 3:
        return
    mu = x[nsol + 1::3] + x[nsol + 2::3] - 2.0 * v
    rm, rc = mu.square().sum(1).sqrt(), b
    mu, cu = mu / rm[:, None], v / rc[:, None]
    scp = (mu * cu).sum(1).clamp(-1.0, 1.0)
    th = torch.acos(scp)
    rout, dr, cstb = par["wshell_rout"], par["wshell_dr"], par["wshell_cstb"]
    shell = torch.zeros(len(rc), dtype=torch.long, device=x.device)
    for k in range(1, nsh):
        shell[rc <= rout[k]] = k
    shell[rc <= rout[nsh - 1] - dr[nsh - 1]] = -1
    for k in range(nsh):
        m = (shell == k).nonzero()[:, 0]
        if not len(m):
            continue
        rank = torch.empty(len(m), dtype=torch.float64, device=x.device)
        rank[torch.sort(th[m], stable=True)[1]] = torch.arange(1, len(m) + 1, dtype=torch.float64, device=x.device)
        t0 = torch.acos(1.0 + (1.0 - 2.0 * rank) / len(m))
        t0 = (t0 - 1.5 * torch.sin(t0) * float(cstb[k])).clamp(0.0, math.pi)
        dth = th[m] - t0 + float(np.atleast_1d(par["wshell_theta_corr"])[k])
        E["water_pol"] = E["water_pol"] + (0.5 * par["fkwpol"] * dth * dth).sum()
        f0 = -par["fkwpol"] * dth / torch.sin(th[m]).clamp_min(1e-10)
        av = cu[m] - mu[m] * scp[m, None]
        d[nsol + 3 * m] += f0[:, None] * (-2.0 * av / rm[m, None] + (mu[m] - cu[m] * scp[m, None]) / rc[m, None])
        for h in (1, 2):
            d[nsol + 3 * m + h] += f0[:, None] * av / rm[m, None]


def _exact_adjoint(s, frames):
    """Per frame, state and Q-atom: derivatives by its charge and LJ factors and its share of the energies."""
    n, a = s.n, s.a
    nat, nsol, sa, nq, ns = n["natom"], n["nat_solute"], n["solv_atom"], n["nqat"], n["nstates"]
    md = s.md
    t = synth.q_tangents(md["qctx"], md["qcrg"], md["qA"], md["qB"])
    P = {k: _t(v).flatten() for k, v in t.items()}
    for k in ("A", "B", "el", "sc", "set"):
        P["qp_" + k], P["qq_" + k] = _t(a["qp_" + k]), _t(a["qq_" + k])
        if k != "set":
            P["qw_" + k] = _t(a["qw_" + k])
    con, isq = _t(a["qconn3"])[:nsol] != 0, _ti(a["iqatom"])[:nsol] > 0
    out = torch.zeros(len(frames), ns, nq, 7, dtype=torch.float64, device=con.device)
    iqs = _ti(a["iqseq"])[:nq]
    for f, x in enumerate(map(_t, frames)):
        u2 = (x[None, :, :] - x[iqs][:, None, :]).square().sum(-1)
        for st in range(ns):
            def tab(name, lead):
                return P[name][:ns * lead * nq].view(ns, -1)[st]

            def sums(r2, on, A, B, q, sc, tq, tA, tB, is14, share):
                i6 = 1.0 / (r2 ** 3 + sc)
                z = lambda v: torch.where(on, v, torch.zeros_like(v)).sum(1)  # noqa: E731
                gA, gB = tA * i6 * i6, -tB * i6
                w = is14 != 0
                out[f, st] += torch.stack([z(tq / r2.sqrt()), z(gA * ~w), z(gB * ~w), z(gA * w), z(gB * w),
                                           z(share * q / r2.sqrt()), z(share * (A * i6 * i6 - B * i6))], 1)

            one = torch.ones((), dtype=torch.float64, device=x.device)
            v = {k: tab("qp_" + k, nsol).view(nq, nsol) for k in ("A", "B", "el", "sc", "set", "dq", "dA", "dB", "is14")}
            on = ~con[None, :] | ((v["set"] != 0) & (con & ~isq)[None, :])
            sums(torch.where(on, u2[:, :nsol], one), on, v["A"], v["B"], v["el"], v["sc"], v["dq"], v["dA"], v["dB"],
                 v["is14"], one)
            for k in range(sa):
                w = {m: tab("qw_" + m, sa).view(sa, nq)[k][:, None] for m in ("A", "B", "el", "sc", "dq", "dA", "dB")}
                lj = 1.0 if k == 0 or not n["solvent_spc"] else 0.0
                r2 = u2[:, nsol + k::sa]
                sums(r2, torch.ones_like(r2, dtype=torch.bool), lj * w["A"], lj * w["B"], w["el"], w["sc"], w["dq"],
                     lj * w["dA"], lj * w["dB"], torch.zeros_like(r2), one)
            v = {k: tab("qq_" + k, nq).view(nq, nq) for k in ("A", "B", "el", "sc", "set", "is14")}
            r2 = u2[:, iqs]
            r2 = torch.where(r2 > 0, r2, torch.ones_like(r2))
            for side, flip in (("i", True), ("j", False)):
                # tables are [jq][iq]; the pair's first atom is the column
                m = {k: (tab("qq_%s_%s" % (k, side), nq).view(nq, nq)) for k in ("dq", "dA", "dB")}
                T = (lambda y: y.T) if flip else (lambda y: y)
                sums(r2, T(v["set"]) != 0, T(v["A"]), T(v["B"]), T(v["el"]), T(v["sc"]), T(m["dq"]), T(m["dA"]),
                     T(m["dB"]), T(v["is14"]), one if flip else 0.0 * one)
    return out.cpu().numpy()


def _exact_fep(case, seed):
    V, lam, r, p = _series(case, seed)
    kT, skip, nb = p["kT"], p["nskip"], p["nbins"]
    nw = len(V)
    V = [v[skip:] + p["alpha"] for v in V]
    r = [y[skip:] for y in r]
    H = [p["A"] * np.exp(-p["mu"] * (y - p["r0"]) - p["eta"] * (y - p["r0"]) ** 2) for y in r]
    vg = [0.5 * (v.sum(1)) - 0.5 * np.sqrt((v[:, 0] - v[:, 1]) ** 2 + 4.0 * h * h) for v, h in zip(V, H)]
    c1 = [1.0 / (1.0 + ((e - v[:, 0]) / h) ** 2) for e, v, h in zip(vg, V, H)]
    gap = [v @ p["coeff"] for v in V]
    step = lambda i, o: -kT * np.log(np.mean(np.exp(-(V[i] @ lam[o] - V[i] @ lam[i]) / kT)))  # noqa: E731
    dgf = np.array([step(i, i + 1) for i in range(nw - 1)])
    dgr = np.array([step(i, i - 1) for i in range(1, nw)])
    dG = np.concatenate([[0.0], np.cumsum(0.5 * (dgf - dgr))])
    lo, hi = min(y.min() for y in gap), max(y.max() for y in gap)
    dGg, cc, npts = np.full((nw, nb), np.nan), np.full((nw, nb), np.nan), np.zeros((nw, nb), np.int32)
    rr = np.full((nw, nb), np.nan)
    for i in range(nw):
        at = ((gap[i] - lo) / ((hi - lo) / nb)).astype(int)
        e = vg[i] - V[i] @ lam[i]
        for k in range(nb):
            m = at == k
            npts[i, k] = m.sum()
            if npts[i, k] > 0 and npts[i, k] >= p["nmin"]:
                av = e[m].mean()
                dGg[i, k] = dG[i] - kT * np.log(np.mean(np.exp(-(e[m] - av) / kT))) + av
                cc[i, k], rr[i, k] = c1[i][m].mean(), r[i][m].mean()
    kept = ~np.isnan(dGg)
    w = np.where(kept, npts, 0)
    tot = w.sum(0)

    def mean(y):
        return np.where((tot > 0) & (tot >= p["nmin"]), (np.where(kept, y, 0.0) * w).sum(0) / np.maximum(tot, 1), np.nan)

    return dict(dgf=dgf, dgr=dgr, dG=dG, gap_range=np.array([lo, hi]), dGg=dGg, c1=cc, npts=None, binned=mean(dGg),
                binned_c1=mean(cc), binned_r=mean(rr), ptsum=None)
