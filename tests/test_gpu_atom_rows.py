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
