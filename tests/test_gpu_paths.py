"""The kernels that a size or a step chooses between, at the sizes where the
choice or a tile changes.

* An MD step in one force launch (few receivers) and in separate ones (more
  than 10,240 receivers in all instances), with the per-atom terms inside the
  integrator (steps that record no energies) and in a pass of their own: FP64
  trajectories of 25 steps.  The paths differ in the order of FP64 sums, 1e-16
  of a force, which 25 steps of 1 fs amplify by less than 1e3; 1e-9 A, the
  bound that graph replay is held to, leaves 1e4.
* Free-energy sums over frames staged 512 and 1,024 at a time, bins 256 at a
  time, windows 64 at a time: counts equal, values within 1e-9 of the host's
  (test_gpu_fep).
* Charge groups of more than 128 atoms (atom-list batches of another size),
  against the oracle with the bounds of test_gpu_shapes; the LRF tensors within
  1e-10 (FP64) and 1e-5 (FP32 pair terms) of the largest of their rank.
* Polarisation shells of more than 1,024 members and members with exactly equal
  angles (waters and their images through the centre), against the oracle.
"""
import numpy as np
import pytest

from oracle.oracle import Oracle
from q6_amd import abi, fep, synth

pytestmark = pytest.mark.gpu


def trajectory(s, v, n, ene_every, steps=25):
    from q6_amd.md import BatchMD
    lam = np.array([0.4, 0.6])
    b = BatchMD([s] * n, [lam] * n, [v] * n, nbcycle=10, ene_every=ene_every, max_frames=steps + 1)
    b.run(steps, graph=False)
    b.sync()
    out = [b.state(k) for k in (0, n - 1)]
    b.close()
    return out


def test_step_paths_agree():
    s = synth.build(13.0, 60, 5, 1, 2, seed=31, chain_region=8.0, q_sigma=0.4, lambdas=[0.4, 0.6], cut=8.0,
                    name="paths")
    v = synth.maxwell_velocities(s, 300.0, 7)
    receivers = 4 * s.n["ncgp_solute"] + s.n["nwat"]
    n = 10240 // receivers + 1
    print(f"\n[gpu] {synth.describe(s)}; {receivers} receivers, {n} instances", flush=True)
    ref = trajectory(s, v, 1, 10)[0]
    for m, every in ((1, 1), (n, 10), (n, 1)):
        for x, vel in trajectory(s, v, m, every):
            assert np.max(np.abs(x - ref[0])) <= 1e-9, (m, every)
            assert np.max(np.abs(vel - ref[1])) <= 1e-7 * np.max(np.abs(ref[1])), (m, every)


@pytest.mark.parametrize("nw,npts,nskip,nbins", [(2, 6, 5, 3), (3, 517, 5, 300), (3, 518, 5, 7), (4, 1030, 5, 12),
                                                 (66, 64, 0, 20), (9, 1025, 1, 257)])
def test_free_energy_tiles(nw, npts, nskip, nbins):
    from q6_amd.md import free_energy
    print(f"\n[gpu] free energy: {nw} windows, {npts} frames, {nskip} skipped, {nbins} bins", flush=True)
    rng = np.random.default_rng(nw + npts)
    lam = np.linspace(1, 0, nw)
    lams = np.stack([lam, 1 - lam], 1)
    V = [np.stack([rng.normal(-20 + 30.0 * i / nw, 2.5, npts), rng.normal(10 - 25.0 * i / nw, 2.5, npts)], 1)
         for i in range(nw)]
    rkl = [rng.uniform(2.0, 4.5, npts) for _ in range(nw)]
    kT, A, mu, eta, r0 = 0.596, 35.0, 0.6, 0.05, 2.0
    coeff = np.array([1.0, -1.0])
    d = free_energy(V, lams, kT, rkl=rkl, nskip=nskip, nbins=nbins, nmin=1, coeff=coeff, A=A, mu=mu, eta=eta, r0=r0)
    dgf, dgr, dG = fep.zwanzig(V, lams, kT, nskip)
    H = [fep.offdiag_coupling(r, A, mu, eta, r0) for r in rkl]
    h = fep.evb_pmf(V, lams, H, kT, coeff, nbins, 1, nskip, rkl=rkl)
    assert np.array_equal(d["npts"], h["npts"]) and np.array_equal(d["ptsum"], h["ptsum"])
    for a, b in ((d["dgf"], dgf), (d["dgr"], dgr), (d["dG"], dG), (d["dGg"], h["dGg"]), (d["dGv"], h["dGv"]),
                 (d["c1"], h["c1"]), (d["binned"], h["binned"]), (d["binned_c1"], h["binned_c1"])):
        a, b = np.asarray(a, float), np.asarray(b, float)
        assert np.array_equal(np.isnan(a), np.isnan(b))
        m = ~np.isnan(a)
        assert np.all(np.abs(a[m] - b[m]) <= 1e-9 * np.maximum(1.0, np.abs(b[m])))


@pytest.mark.parametrize("precision,dtol,etol,ltol", [(abi.QNB_PREC_FP64, 1e-10, 1e-10, 1e-10),
                                                      (abi.QNB_PREC_MIXED, 5e-6, 1e-5, 1e-5)])
@pytest.mark.parametrize("chains,beads", [(2, 150), (2, 129), (3, 128)])
def test_large_groups_and_lrf(chains, beads, precision, dtol, etol, ltol):
    from q6_amd.engine import NonbondedEngine
    s = synth.build(17.0, chains, beads, 1, 2, seed=chains + beads, chain_region=13.0, q_sigma=0.4,
                    lambdas=[0.3, 0.7], cut=8.0, q_per_chain=9, name="large-groups")
    print(f"\n[gpu] {synth.describe(s)} precision {precision}", flush=True)
    o = Oracle(s)
    o.make_pair_lists(s.x)
    do, Eo, _ = o.eval_terms(abi.T_ALL, s.x, Tfree=300.0)
    eng = NonbondedEngine(s, precision=precision)
    eng.make_pair_lists(s.x)
    d, E, _ = eng.eval_terms(abi.T_ALL, s.x, Tfree=300.0)
    assert np.max(np.abs(d - do)) <= dtol * np.max(np.abs(do))
    e, eo = (np.array([q[k] for k in ("ww_el", "pw_el", "pw_vdw", "pp_el", "pp_vdw", "lrf")]) for q in (E, Eo))
    assert np.max(np.abs(e - eo)) <= etol * np.max(np.abs(eo))
    L, Lo = eng.lrf(), o.lrf().reshape(-1, 43)
    for lo, hi in ((3, 4), (4, 7), (7, 16), (16, 43)):
        assert np.max(np.abs(L[:, lo:hi] - Lo[:, lo:hi])) <= ltol * np.max(np.abs(Lo[:, lo:hi])), (lo, hi)
    eng.close()


@pytest.mark.parametrize("radius", [9.0, 31.0])
def test_polarisation_ranks(radius):
    from q6_amd.engine import NonbondedEngine
    s = synth.build(radius, 0, 1, 0, 1, seed=41, chain_region=0.5 * radius, lambdas=[1.0], cut=7.0,
                    water_fill=radius, name="shells")
    if radius > 20.0:
        s.par["wshell_dr"][-1] = 7.0  # the innermost shell's 2,000 or so members
    nw = s.n["nwat"]
    x = s.x.copy()
    half = nw // 2
    x[3 * half:6 * half] = -x[:3 * half]  # equal angles, in pairs (the sphere's centre is the origin)
    print(f"\n[gpu] {synth.describe(s)}: {half} pairs of equal angles", flush=True)
    mask = abi.T_RAD | abi.T_POL
    o = Oracle(s)
    o.make_pair_lists(x)
    eng = NonbondedEngine(s, precision=abi.QNB_PREC_FP64)
    eng.make_pair_lists(x)
    for step in range(2):  # the second call finds the first one's shell state
        do, Eo, _ = o.eval_terms(mask, x, Tfree=300.0, istep=step)
        d, E, _ = eng.eval_terms(mask, x, Tfree=300.0, istep=step)
        assert np.max(np.abs(d - do)) <= 1e-10 * np.max(np.abs(do))
        for k in ("solvent_radial", "water_pol"):
            assert abs(E[k] - Eo[k]) <= 1e-10 * max(abs(Eo[k]), 1e-12), k
        assert np.allclose(eng.shell_state(), o.shell_state(), rtol=1e-10, atol=1e-12)
    eng.close()
