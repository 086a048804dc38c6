"""Every term of one evaluation against the oracle at the sizes where a launch
shape can go wrong: fewer charge groups than the energy reduction has waves,
a few waters, mostly solute, no solute, groups larger than a receiver sweep, 1 to 4
states.

FP64: gradients and energies are sums of at most a few thousand terms whose
order differs from the oracle's, so each is within 1e-12 of the largest
component (n eps with n ~ 4e3); the suite's general bound of 1e-10 is used for
cancellation between terms.  Mixed: the pair arithmetic's FP32 rounding, the
bounds of test_gpu_configs (5e-6 of the largest gradient component, 1e-5 of the
largest energy).
"""
import numpy as np
import pytest

from oracle.oracle import Oracle
from q6_amd import abi, synth

pytestmark = pytest.mark.gpu

# radius, chains, beads, Q chains, states, Q-atoms per chain
SHAPES = {
    "few_waters": (5.0, 1, 4, 1, 1, None),
    "no_solute": (8.0, 0, 1, 0, 1, None),
    "mostly_solute": (9.0, 19, 7, 1, 2, 3),
    "large_groups": (13.0, 3, 23, 1, 2, 11),
    "many_groups": (14.0, 60, 5, 3, 4, None),
}


def system(key):
    r, nc, nb, nqc, ns, qpc = SHAPES[key]
    return synth.build(r, nc, nb, nqc, ns, seed=23, chain_region=0.5 * r, q_sigma=0.4,
                       lambdas=np.arange(1, ns + 1) / (ns * (ns + 1) / 2), cut=7.0, q_per_chain=qpc,
                       water_fill=r, name=key)


def flat(E, EQ):
    out = [E[k] for k in ("ww_el", "ww_vdw", "pw_el", "pw_vdw", "pp_el", "pp_vdw", "lrf", "solvent_radial",
                          "water_pol")]
    for q in EQ:
        out += [q["qq_el"], q["qq_vdw"], q["qp_el"], q["qp_vdw"], q["qw_el"], q["qw_vdw"]]
    return np.array(out)


@pytest.mark.parametrize("key", list(SHAPES))
@pytest.mark.parametrize("precision,dtol,etol", [(abi.QNB_PREC_FP64, 1e-10, 1e-10), (abi.QNB_PREC_MIXED, 5e-6, 1e-5)])
def test_evaluation_matches_oracle(key, precision, dtol, etol):
    from q6_amd.engine import NonbondedEngine
    s = system(key)
    print(f"\n[gpu] {synth.describe(s)} precision {precision}", flush=True)
    o = Oracle(s)
    o.make_pair_lists(s.x)
    do, Eo, EQo = o.eval_terms(abi.T_ALL, s.x, Tfree=300.0)
    eng = NonbondedEngine(s, precision=precision)
    eng.make_pair_lists(s.x)
    for _ in range(2):  # the second call finds what the first one left behind
        d, E, EQ = eng.eval_terms(abi.T_ALL, s.x, Tfree=300.0)
        assert np.max(np.abs(d - do)) <= dtol * max(np.max(np.abs(do)), 1e-12)
        e, eo = flat(E, EQ), flat(Eo, EQo)
        assert np.max(np.abs(e - eo)) <= etol * max(np.max(np.abs(eo)), 1e-12)
    eng.close()
