"""Atoms whose coordinates no single FP32 step brings back into the box (an atom that left, a
trajectory that blew up), on every path from binning to the displaced atoms.  They carry no
charge and no epsilon, so the others' energies, forces and pairs are those without them."""
import dataclasses

import numpy as np
import pytest

from atmmetaforce import ATMBatch, workloads as W
from oracle import oracle

pytestmark = pytest.mark.gpu

FAR = ([3e7, -2e8, 5e9], [-7e12, 4e4, -1e10], [2e38, -2e38, 2e38], [1.0, 2.0, -6e37])


def _systems(tilt):
    p = W.ATMParams(0.2, 0.4, 0.1, 110.0, 0.0, 200.0, 100.0, 0.0625, 1.0)
    s = W.lattice_system(1500, 3.5, 0.9, 30, (0.875, 0.875, 0.875), 41, p)
    if tilt is not None:
        s.tilt = np.array(tilt)
    n = s.num_atoms
    moved = int(np.argmax(np.any(s.displacements != 0.0, axis=1)))
    at = np.array([5, moved, n // 2, moved + 1])  # two of them among the displaced atoms
    far = dataclasses.replace(s, positions=s.positions.copy(), charges=s.charges.copy(), epsilons=s.epsilons.copy())
    far.positions[at], far.charges[at], far.epsilons[at] = FAR, 0.0, 0.0
    keep = np.setdiff1d(np.arange(n), at)
    near = dataclasses.replace(far, **{k: getattr(far, k)[keep] for k in
                                       ("positions", "charges", "sigmas", "epsilons", "displacements")})
    return far, near, at, keep


@pytest.mark.parametrize("tilt", [None, (0.875, -0.75, 1.125)])
@pytest.mark.parametrize("full_state2", [False, True])
def test_far_positions(gpu, tilt, full_state2):
    far, near, at, keep = _systems(tilt)
    ref, Fref = oracle.atm_eval(near)
    print(f"[far] tilt {tilt} full {full_state2}", flush=True)
    with ATMBatch([far]) as b:
        b.set_tuning(full_state2=full_state2)
        for mode in (dict(), dict(plain=True), dict(forces=False), dict(forces=False, param_grads=True), dict(fp32_pairs=True)):
            print(f"[far] {mode}", flush=True)
            b.compute(**mode)
            r = b.result(0)
            # FP64 pair energies in another order: 1e-13 of the sum of their magnitudes (FP32: 2^-24 each)
            assert abs(r["state1_energy"] - ref["U1"]) <= (1e-6 if "fp32_pairs" in mode else 1e-13) * max(ref["abs1"], 1.0)
            if mode.get("forces", True) and "fp32_pairs" not in mode:
                F = b.forces(0)
                # FP32 force vectors (2^-24 each) and per-lane sums of up to ~100 of them
                assert np.linalg.norm(F[keep] - Fref) <= 1e-6 * np.linalg.norm(Fref)
                assert not F[at].any()
        b.compute()
        for st in (0, 1):  # the pairs of the other atoms are found as without the far ones
            got = b.pairs(0, st)
            got = got[~np.isin(got, at).any(1)]
            want = keep[oracle.pairs(near.positions + (near.displacements if st else 0.0), near.box, near.cutoff, tilt=near.tilt)]
            assert np.array_equal(got, want)
