"""Partner-atom rows of the receivers: their memory and their growth.

* Memory: a batch's rows follow the longest row of its systems (half as many
  slots again, or a cut-off sphere of solute), not the solute's size times the
  number of groups.  1,500 solute atoms in 150 ten-atom groups at a cut-off of
  7 A: the longest row holds 110 atoms, so its rows and the neighbour rows fit
  the 1,024 numbers of 4 bytes that the first list build has for each of the
  2,166 groups, 9 MB, and at most 7 MB are left for everything else of an
  instance (44 numbers per group and 65 per atom, of 8 bytes); rows for all
  solute atoms alone would take 26.5 MB.
* Growth: rows longer than the slots an engine starts with (a cut-off sphere of
  solute, 256 slots at 5.2 A; two groups of 140 atoms take 320; seed 1 has such
  rows, seed 2 none), against the oracle with the bounds of test_gpu_shapes,
  before and after a second list update.
* Rows that outgrow a batch's space in a run: eight chains of 100 (140) atoms
  without LJ fly together from 30 A apart, where every row is empty and gets the
  256 slots of a cut-off sphere; together a row holds 700 (980) atoms, of which
  200 (none) are stored.  From there on the run is compared with a batch created on
  the same positions, whose rows hold everything: FP64 within the bounds of
  test_gpu_paths; mixed velocities of solute atoms within n 5e-6 dmax w dt of
  each other for n steps (test_gpu_branches), in one launch and in separate kernels.
"""
import ctypes as C

import numpy as np
import pytest

from oracle.oracle import Oracle
from q6_amd import abi, synth

pytestmark = pytest.mark.gpu


def test_memory_of_a_batch():
    from q6_amd.md import BatchMD
    s = synth.build(28.0, 150, 10, 1, 2, seed=17, chain_region=18.0, q_sigma=0.4, lambdas=[0.4, 0.6], cut=7.0)
    n = 16
    print(f"\n[gpu] {synth.describe(s)}: memory of {n} instances", flush=True)
    v = synth.maxwell_velocities(s, 300.0, 7)

    def free():
        left, total = C.c_size_t(), C.c_size_t()
        assert abi.load().hipMemGetInfo(C.byref(left), C.byref(total)) == 0  # of the runtime the library uses
        return left.value

    def held(n):
        before = free()
        b = BatchMD([s] * n, [np.array([0.4, 0.6])] * n, [v] * n, precision=abi.QNB_PREC_MIXED, max_frames=1)
        after = free()
        b.close()
        return before - after

    held(1)
    per = (held(n) - held(1)) / (n - 1) / 1e6
    print(f"{per:.1f} MB per instance, {s.n['ncgp']} groups", flush=True)
    assert per < 16.0


@pytest.mark.parametrize("precision,dtol,etol", [(abi.QNB_PREC_FP64, 1e-10, 1e-10), (abi.QNB_PREC_MIXED, 5e-6, 1e-5)])
@pytest.mark.parametrize("seed", [1, 2])
def test_rows_longer_than_the_first_slots(seed, precision, dtol, etol):
    from q6_amd.engine import NonbondedEngine
    s = synth.build(20.0, 8, 140, 1, 2, seed=seed, chain_region=16.0, q_sigma=0.4, lambdas=[0.3, 0.7], cut=5.2,
                    q_per_chain=9)
    print(f"\n[gpu] {synth.describe(s)} precision {precision}: rows grow", flush=True)
    eng = NonbondedEngine(s, precision=precision)
    rng = np.random.default_rng(seed)
    for x in (s.x, s.x + rng.normal(0.0, 0.02, s.x.shape)):
        o = Oracle(s)
        o.make_pair_lists(x)
        do, Eo, _ = o.eval_terms(abi.T_ALL, x, Tfree=300.0)
        eng.make_pair_lists(x)
        d, E, _ = eng.eval_terms(abi.T_ALL, x, Tfree=300.0)
        assert np.max(np.abs(d - do)) <= dtol * np.max(np.abs(do))
        e, eo = (np.array([q[k] for k in ("ww_el", "pw_el", "pw_vdw", "pp_el", "pp_vdw", "lrf")]) for q in (E, Eo))
        assert np.max(np.abs(e - eo)) <= etol * np.max(np.abs(eo))
    eng.close()


@pytest.mark.parametrize("precision", [abi.QNB_PREC_FP64, abi.QNB_PREC_MIXED])
@pytest.mark.parametrize("beads", [100, 140])
def test_rows_that_outgrow_a_batch(beads, precision):
    from q6_amd.engine import NonbondedEngine
    from q6_amd.md import BatchMD
    chains, inbound, steps, dt = 8, 10, 3, 0.020462
    s = synth.build(24.0, chains, beads, 1, 2, seed=5, chain_region=19.0, q_sigma=0.2, lambdas=[0.3, 0.7], cut=5.2,
                    q_per_chain=3, water_fill=9.0, use_lrf=False)
    n = s.n["nat_solute"]
    for k in ("avdw", "bvdw", "pw_A", "pw_B", "qp_A", "qp_B", "qw_A", "qw_B"):
        s.a[k] = np.zeros_like(s.a[k])  # atoms pass through one another
    s.a["crg"][:n] *= 0.1
    for k in ("pw_el", "qp_el", "qw_el"):
        s.a[k] = s.a[k] * 0.01
    s.par["fk_wsphere"] = s.par["Dwmz"] = 0.0  # its radius follows the temperature, which flying chains raise
    rng = np.random.default_rng(beads)
    of = np.arange(n) // beads
    sw = s.a["cgp_iswitch"][:chains]
    away = np.stack([[(k & 1) * 2 - 1, (k >> 1 & 1) * 2 - 1, (k >> 2) * 2 - 1] for k in range(chains)]) * 30.0
    x, v = s.x.copy(), np.zeros_like(s.x)
    x[:n] += (rng.normal(0.0, 1.0, (chains, 3)) - s.x[sw] + away)[of]
    v[:n] = (-away / (inbound * dt))[of]

    def batch(count, x, v):
        return BatchMD([s] * count, [np.array([0.3, 0.7])] * count, [v] * count, precision=precision, nbcycle=1,
                       ene_every=10, max_frames=20, tau_T_fs=1e9, positions=[x] * count)

    per = 4 * chains + s.n["nwat"]
    print(f"\n[gpu] {synth.describe(s)} precision {precision}: {chains} chains fly together", flush=True)
    for count in (1, 10240 // per + 1):
        a = batch(count, x, v)
        a.run(inbound, graph=False)
        a.sync()
        xa, va = a.state(count - 1)
        assert np.max(np.linalg.norm(xa[sw], axis=1)) < 5.2
        b = batch(count, xa, va)
        for c in (a, b):
            c.run(steps, graph=False)
            c.sync()
        (x1, v1), (x2, v2) = a.state(count - 1), b.state(count - 1)
        a.close()
        b.close()
        if precision == abi.QNB_PREC_FP64:
            assert np.max(np.abs(x1 - x2)) <= 1e-9 and np.max(np.abs(v1 - v2)) <= 1e-7 * np.max(np.abs(v2)), count
        else:
            eng = NonbondedEngine(s)
            eng.make_pair_lists(xa)
            dmax = np.max(np.abs(eng.eval_terms(abi.T_ALL, xa, Tfree=300.0)[0]))
            eng.close()
            dv = np.abs(v1 - v2)[:n]
            assert np.all(dv <= (2 * steps * 5e-6 * dmax * dt / np.asarray(s.md["mass"])[:n])[:, None]), count
