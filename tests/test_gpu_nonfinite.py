"""Coordinates without a finite answer: what such a call reports, and that it
leaves the rest of its results and the next call alone.

* A water of a polarisation shell whose dipole has no direction (its hydrogens
  not a number): every call reports a non-finite energy, the other waters'
  gradients stay finite, and the next call on finite coordinates equals the
  oracle (1e-10, the bound of test_gpu_paths).
* A frame with a water that is not a number: the adjoint's sums over the waters
  of that frame are not numbers, those of the other frames are unchanged.
* Two atoms in one place and an atom 1e160 A away, whose squared distances are 0
  and infinite: infinite sums where the enumeration in numpy has them, finite
  ones beside them (1e-10; FP32 pairs 5e-6 of the largest of their kind, the
  bound of test_gpu_shapes); the far atom adds nothing to an FP64 evaluation
  (in FP32 its position itself is infinite).
"""
import numpy as np
import pytest

from adjoint_ref import slot_sums
from oracle.oracle import Oracle
from q6_amd import abi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lost", [1, 3])
def test_polarisation_angle_not_a_number(lost):
    from q6_amd.engine import NonbondedEngine
    s = synth.build(9.0, 0, 1, 0, 1, seed=41, chain_region=4.5, lambdas=[1.0], cut=7.0, water_fill=9.0, name="shells")
    mask = abi.T_RAD | abi.T_POL
    x = s.x.copy()
    out = np.argsort(np.linalg.norm(x[::3], axis=1))[-lost:]  # waters of the outermost shell
    for w in out:
        x[3 * w + 1:3 * w + 3] = np.nan
    print(f"\n[gpu] {synth.describe(s)}: hydrogens of {lost} waters not a number", flush=True)
    eng = NonbondedEngine(s, precision=abi.QNB_PREC_FP64)
    eng.make_pair_lists(s.x)
    state = eng.shell_state()
    for _ in range(5):
        d = np.zeros_like(x)
        with pytest.raises(abi.QnbError, match="non-finite"):
            eng.eval_terms(mask, x, Tfree=300.0, d=d)
        lostatoms = np.isin(np.arange(len(x)) // 3, out)
        assert np.all(np.isfinite(d[~lostatoms])) and np.all(np.isnan(d[lostatoms]).any(1))
        eng.set_shell_state(state)
    o = Oracle(s)
    o.make_pair_lists(s.x)
    do, Eo, _ = o.eval_terms(mask, s.x, Tfree=300.0)
    d, E, _ = eng.eval_terms(mask, s.x, Tfree=300.0)
    assert np.max(np.abs(d - do)) <= 1e-10 * np.max(np.abs(do))
    assert abs(E["water_pol"] - Eo["water_pol"]) <= 1e-10 * abs(Eo["water_pol"])
    assert np.allclose(eng.shell_state(), o.shell_state(), rtol=1e-10, atol=1e-12)
    eng.close()


def nine_site():
    s = synth.build(13.0, 3, 6, 1, 2, 41, chain_region=5.0, q_sigma=0.4, lambdas=[0.4, 0.6], water_fill=12.0)
    return synth.replace_solvent(s, synth.ethanol(), 0.0085, 48)


@pytest.mark.parametrize("precision", [abi.QNB_PREC_FP64, abi.QNB_PREC_MIXED])
@pytest.mark.parametrize("build", [lambda: synth.build(11.0, 4, 8, 2, 2, seed=5, chain_region=5.0, q_sigma=0.4,
                                                       lambdas=[0.3, 0.7], cut=7.0, q_per_chain=4), nine_site],
                         ids=["water", "nine_site"])
def test_adjoint_of_a_lost_water(build, precision):
    from q6_amd import adjoint
    from q6_amd.engine import NonbondedEngine
    s = build()
    frames = np.stack([s.x] * 3)
    frames[1, s.n["nat_solute"]:s.n["nat_solute"] + s.n["solv_atom"]] = np.nan
    print(f"\n[gpu] {synth.describe(s)} precision {precision}: first solvent molecule of frame 1 lost", flush=True)
    tangent, _keep = adjoint.tangent_struct(s)
    eng = NonbondedEngine(s, precision=precision)
    out = eng.adjoint(tangent, frames)
    eng.close()
    assert np.all(np.isfinite(out[[0, 2]])) and np.array_equal(out[0], out[2])
    assert np.all(np.isnan(out[1][..., [abi.ADJ_DQ, abi.ADJ_DA, abi.ADJ_DB, abi.ADJ_EEL, abi.ADJ_EVDW]]))


def limits_case():
    s = synth.build(11.0, 4, 8, 2, 2, seed=5, chain_region=5.0, q_sigma=0.4, lambdas=[0.3, 0.7], cut=7.0, q_per_chain=4)
    a = s.a
    away = [j for j in range(s.n["nat_solute"]) if not a["qconn3"][j] and j not in a["cgp_iswitch"]]
    same, far = s.x.copy(), s.x.copy()
    same[away[-1]] = s.x[a["iqseq"][0]]
    far[away[-1], 0] = 1e160
    return s, same, far


@pytest.mark.parametrize("precision,tol", [(abi.QNB_PREC_FP64, 1e-10), (abi.QNB_PREC_MIXED, 5e-6)])
def test_adjoint_at_the_limits_of_a_distance(precision, tol):
    from q6_amd import adjoint
    from q6_amd.engine import NonbondedEngine
    s, same, far = limits_case()
    print(f"\n[gpu] {synth.describe(s)} precision {precision}: an atom on a Q-atom; one far away", flush=True)
    tangent, _keep = adjoint.tangent_struct(s)
    eng = NonbondedEngine(s, precision=precision)
    out = eng.adjoint(tangent, np.stack([same, far]))
    eng.close()
    tang = synth.q_tangents(s.md["qctx"], s.md["qcrg"], s.md["qA"], s.md["qB"])
    with np.errstate(all="ignore"):
        ref = np.stack([slot_sums(s, x, tang) for x in (same, far)])
    assert np.isinf(ref[0]).any() and np.all(np.isfinite(ref[1]))
    assert np.array_equal(np.isnan(out), np.isnan(ref))
    assert np.array_equal(np.where(np.isinf(out), out, 0.0), np.where(np.isinf(ref), ref, 0.0))
    m = np.isfinite(ref)
    for c in range(abi.QNB_ADJ_NV):
        o, r = out[..., c][m[..., c]], ref[..., c][m[..., c]]
        assert np.max(np.abs(o - r)) <= tol * np.max(np.abs(r)), c


def test_evaluation_with_a_far_atom():
    from q6_amd.engine import NonbondedEngine
    s, _, far = limits_case()
    print(f"\n[gpu] {synth.describe(s)}: one atom far away", flush=True)
    mask = abi.T_PP | abi.T_PW
    o = Oracle(s)
    o.make_pair_lists(s.x)
    do, Eo, _ = o.eval_terms(mask, far, Tfree=300.0)
    eng = NonbondedEngine(s, precision=abi.QNB_PREC_FP64)
    eng.make_pair_lists(s.x)
    d, E, _ = eng.eval_terms(mask, far, Tfree=300.0)
    eng.close()
    assert np.all(np.isfinite(do)) and np.max(np.abs(d - do)) <= 1e-10 * np.max(np.abs(do))
    e, eo = (np.array([q[k] for k in ("pp_el", "pp_vdw", "pw_el", "pw_vdw")]) for q in (E, Eo))
    assert np.max(np.abs(e - eo)) <= 1e-10 * np.max(np.abs(eo))
