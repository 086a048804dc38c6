"""The force kernels on both sides of the one-launch bound (10,240 receiver
waves in all instances: four per solute group, one per solvent molecule), and
batches of unlike systems.

* One evaluation above the bound, 3-site water and a nine-site solvent, FP64 and
  mixed, against the oracle with the bounds of test_gpu_shapes.
* A mixed MD step in one launch and in separate kernels, with the per-atom terms
  in the integrator and in a pass of their own, against FP64 steps.  A mixed
  gradient is within 5e-6 of the largest component (test_gpu_shapes), so n steps
  move a velocity by at most n 5e-6 dmax w dt; 1e-6 of the largest velocity is
  left for the Berendsen factor.  Solute atoms are compared one by one; SHAKE
  ends its iterations at 1e-4 of a squared bond, which another rounding reaches
  an iteration later, so a water is compared by its momentum, which the
  constraints leave alone, and by its positions within 1e-4 A.
* A batch of systems that differ in size, states, Q-atoms, list rule and LRF, in
  one launch and in separate kernels: each member as in a batch of its own, FP64
  25 steps within the bounds of test_gpu_paths.
"""
import numpy as np
import pytest

from oracle.oracle import Oracle
from q6_amd import abi, synth

pytestmark = pytest.mark.gpu

DT = 0.020462


def receivers(s):
    return 4 * s.n["ncgp_solute"] + s.n["nwat"]


def water_above():
    return synth.build(43.5, 12, 10, 2, 3, seed=61, chain_region=14.0, q_sigma=0.4, lambdas=[0.2, 0.3, 0.5], cut=6.5,
                       rclrf=9.0, q_per_chain=6)


def nine_above():
    s = synth.build(36.0, 2600, 2, 2, 2, 62, chain_region=33.0, q_sigma=0.4, lambdas=[0.4, 0.6], cut=6.5, rclrf=9.0,
                    water_fill=30.0)
    return synth.replace_solvent(s, synth.ethanol(), 0.002, 48)


@pytest.mark.parametrize("precision,dtol,etol", [(abi.QNB_PREC_FP64, 1e-10, 1e-10), (abi.QNB_PREC_MIXED, 5e-6, 1e-5)])
@pytest.mark.parametrize("build", [water_above, nine_above])
def test_evaluation_above_the_bound(build, precision, dtol, etol):
    from q6_amd.engine import NonbondedEngine
    s = build()
    print(f"\n[gpu] {synth.describe(s)} precision {precision}: {receivers(s)} receiver waves", flush=True)
    assert receivers(s) > 10240 and s.n["nwat"] > 0
    o = Oracle(s)
    o.make_pair_lists(s.x)
    do, Eo, EQo = o.eval_terms(abi.T_ALL, s.x, Tfree=300.0)
    eng = NonbondedEngine(s, precision=precision)
    eng.make_pair_lists(s.x)
    for _ in range(2):  # the second call finds what the first one left behind
        d, E, EQ = eng.eval_terms(abi.T_ALL, s.x, Tfree=300.0)
        assert np.max(np.abs(d - do)) <= dtol * np.max(np.abs(do))
        e, eo = (np.array(list(a.values()) + [v for q in b for v in q.values()]) for a, b in ((E, EQ), (Eo, EQo)))
        assert np.max(np.abs(e - eo)) <= etol * np.max(np.abs(eo))
    eng.close()


def run(systems, precision, every, steps):
    from q6_amd.md import BatchMD
    b = BatchMD(systems, [np.asarray(s.par["lambda"], float) for s in systems],
                [synth.maxwell_velocities(s, 300.0, 7) for s in systems], precision=precision, nbcycle=10,
                ene_every=every, max_frames=steps + 1)
    b.run(steps, graph=False)
    b.sync()
    out = [b.state(k) for k in range(len(systems))]
    b.close()
    return out


@pytest.mark.parametrize("every", [1, 10])
def test_mixed_step_paths_agree(every):
    from q6_amd.engine import NonbondedEngine
    s = synth.build(13.0, 60, 5, 1, 2, seed=31, chain_region=8.0, q_sigma=0.4, lambdas=[0.4, 0.6], cut=8.0, name="paths")
    n, steps = 10240 // receivers(s) + 1, 3
    print(f"\n[gpu] {synth.describe(s)}; {receivers(s)} receivers, {n} instances, energies every {every}", flush=True)
    eng = NonbondedEngine(s)
    eng.make_pair_lists(s.x)
    dmax = np.max(np.abs(eng.eval_terms(abi.T_ALL, s.x, Tfree=300.0)[0]))
    eng.close()
    x, v = run([s], abi.QNB_PREC_FP64, 10, steps)[0]
    nsol, mass = s.n["nat_solute"], np.asarray(s.md["mass"], float)
    slack = 1e-6 * np.max(np.abs(v))
    for m in (1, n):
        out = run([s] * m, abi.QNB_PREC_MIXED, every, steps)
        for xm, vm in (out[0], out[-1]):
            dv = np.abs(vm - v)
            assert np.all(dv[:nsol] <= (steps * 5e-6 * dmax * DT / mass[:nsol])[:, None] + slack), m
            mw = mass[nsol:].reshape(-1, 3)
            dp = np.abs((((vm - v)[nsol:].reshape(-1, 3, 3)) * mw[:, :, None]).sum(1)) / mw.sum(1)[:, None]
            assert np.all(dp <= (steps * 3 * 5e-6 * dmax * DT / mw.sum(1))[:, None] + slack), m
            assert np.max(np.abs(xm - x)) <= 1e-4, m


def unlike():
    def build(*a, **k):
        return synth.build(*a, q_sigma=0.4, cut=8.0, **k)
    many = build(14.0, 30, 6, 3, 3, seed=71, chain_region=8.0, lambdas=[0.2, 0.3, 0.5], q_per_chain=4)
    no_q = build(12.0, 8, 5, 0, 1, seed=72, chain_region=6.0, lambdas=[1.0])
    water = build(9.0, 0, 1, 0, 1, seed=73, chain_region=4.0, lambdas=[1.0], water_fill=9.0)
    no_lrf = build(13.0, 12, 9, 1, 2, seed=74, chain_region=7.0, lambdas=[0.4, 0.6], use_lrf=False)
    any_atom = build(12.0, 10, 8, 2, 1, seed=75, chain_region=7.0, lambdas=[1.0])
    any_atom.n["any_atom_cutoff"] = 1
    return [many, no_q, water, no_lrf, any_atom]


@pytest.mark.parametrize("every", [1, 10])
def test_unlike_systems_in_one_batch(every):
    members = unlike()
    total = sum(receivers(s) for s in members)
    print(f"\n[gpu] {[synth.describe(s) for s in members]}; {total} receivers, energies every {every}", flush=True)
    assert total < 10240
    alone = [run([s], abi.QNB_PREC_FP64, every, 25)[0] for s in members]
    for copies in (1, 10240 // total + 1):
        out = run(members * copies, abi.QNB_PREC_FP64, every, 25)
        for k, (x, v) in list(enumerate(out))[:5] + list(enumerate(out))[-5:]:
            xr, vr = alone[k % 5]
            assert np.max(np.abs(x - xr)) <= 1e-9, (copies, k)
            assert np.max(np.abs(v - vr)) <= 1e-7 * np.max(np.abs(vr)), (copies, k)


def test_q_atoms_are_taken_from_iqseq():
    """An evaluation takes the Q-atoms' places from iqseq; iqatom only says
    which atoms they are (a caller may hold plain flags there)."""
    from q6_amd.engine import NonbondedEngine
    s = synth.build(14.0, 60, 5, 3, 4, seed=23, chain_region=7.0, q_sigma=0.4, lambdas=[0.1, 0.2, 0.3, 0.4], cut=7.0)
    print(f"\n[gpu] {synth.describe(s)}: flags for Q-atom numbers", flush=True)
    o = Oracle(s)
    o.make_pair_lists(s.x)
    do, Eo, EQo = o.eval_terms(abi.T_ALL, s.x, Tfree=300.0)
    s.a["iqatom"] = (s.a["iqatom"] > 0).astype(np.int32)
    eng = NonbondedEngine(s, precision=abi.QNB_PREC_FP64)
    eng.make_pair_lists(s.x)
    d, E, EQ = eng.eval_terms(abi.T_ALL, s.x, Tfree=300.0)
    eng.close()
    assert np.max(np.abs(d - do)) <= 1e-10 * np.max(np.abs(do))
    e, eo = (np.array(list(a.values()) + [v for q in b for v in q.values()]) for a, b in ((E, EQ), (Eo, EQo)))
    assert np.max(np.abs(e - eo)) <= 1e-10 * np.max(np.abs(eo))
