"""Batch adjoint over more (frame, Q-atom) pairs than one row of a launch holds.

85,000 frames of 200 Q-atoms are 17.0 million blocks of 256 threads, past the
2^32 threads of a launch along x; every frame's record is the one that the
single-system entry point, which takes 256 frames at a time, returns for it.
"""
import numpy as np
import pytest

from q6_amd import abi, adjoint, synth

pytestmark = pytest.mark.gpu


def test_seventeen_million_blocks():
    from q6_amd.engine import NonbondedEngine
    from q6_amd.md import BatchMD
    s = synth.build(14.0, 20, 10, 20, 1, seed=3, chain_region=12.0, lambdas=[1.0], cut=8.0, water_fill=6.0)
    nq, nf = s.n["nqat"], 85000
    print(f"\n[gpu] {synth.describe(s)}: adjoint over {nf} frames x {nq} Q-atoms", flush=True)
    assert nq == 200
    # steps so short that the unrelaxed start stays where it is
    b = BatchMD([s], [np.ones(1)], [synth.maxwell_velocities(s, 300.0, 5)], precision=abi.QNB_PREC_MIXED, dt_fs=1e-7,
                nbcycle=100, ene_every=100, max_frames=1)
    b.store_frames(1, nf)
    b.run(nf)
    tangent, _keep = adjoint.tangent_struct(s)
    out = b.adjoint([tangent])[0]
    frames = b.frames(0)
    b.close()
    assert out.shape[0] == len(frames) == nf
    # the frames on both sides of every row's end, among others
    rows = -(-nf * nq // (1 << 22))
    ends = [k * -(-nf * nq // rows) // nq for k in range(1, rows)]
    pick = np.unique([0, 1, nf - 2, nf - 1] + [f for e in ends for f in (e - 1, e, e + 1)])
    eng = NonbondedEngine(s, precision=abi.QNB_PREC_MIXED)
    assert np.array_equal(eng.adjoint(tangent, frames[pick]), out[pick])
    eng.close()
    assert np.all(np.isfinite(out)) and np.all(np.abs(out).max((1, 2, 3)) > 0)
