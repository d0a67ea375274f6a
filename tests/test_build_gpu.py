"""Binning and sorting of one set by one block (up to 4,096 atoms) and by the chain of kernels
(above): the two give the same clusters, so the same sums."""
import numpy as np
import pytest

from atmmetaforce import ATMBatch, workloads as W
from oracle import oracle

pytestmark = pytest.mark.gpu

P = W.ATMParams(0.2, 0.4, 0.1, 110.0, 0.0, 200.0, 100.0, 0.0625, 1.0)


def _system(n, L=3.4, tilt=None):
    s = W.lattice_system(n, L, 0.9, max(1, n // 50), (L / 4, L / 4, L / 4), 11 + n, P)
    if tilt is not None:
        s.tilt = np.array(tilt)
    return s


# tilts on the 2^-20 nm grid of the positions, where every wrapping step is exact; (0.9, -0.8, 1.1)
# rounds to FP32 by up to 6e-8 nm, which moved U1 of 63 atoms by 1e-7 kJ/mol
@pytest.mark.parametrize("tilt", [None, (0.875, -0.75, 1.125)])
# less than a wave, the block's width, its second pass, the last size of the one-block path, the first beyond it
@pytest.mark.parametrize("n", [1, 63, 1023, 1025, 2049, 4095, 4096, 4097])
def test_sizes(gpu, n, tilt):
    s = _system(n, tilt=tilt)
    with ATMBatch([s]) as b:
        b.compute()
        r, F = b.result(0), b.forces(0)
        ref, Fref = oracle.atm_eval(s)
        # FP64 pair energies in another order: 1e-13 of the sum of their magnitudes
        assert abs(r["state1_energy"] - ref["U1"]) <= 1e-13 * max(ref["abs1"], 1.0)
        # FP32 force vectors (2^-24 each) and per-lane sums of up to ~100 of them
        assert np.linalg.norm(F - Fref) <= 1e-6 * max(np.linalg.norm(Fref), 1e-3)
        b.compute(forces=False)
        assert b.result(0)["energy"] == pytest.approx(r["energy"], rel=1e-12, abs=1e-12)
        assert not b.forces(0).any()  # an energy evaluation clears the accumulated force


def test_both_routes_the_same(gpu):
    """A small system alone (one block) and beside one of 4,097 atoms (the chain): the sorted
    order is the same and both batches run 16 waves per group, so every sum is, to the last bit."""
    small, large = _system(1500), _system(4097)
    with ATMBatch([small, small]) as a, ATMBatch([small, large]) as b:
        a.compute()
        b.compute()
        assert a.list_stats()["pairs"][0] == b.list_stats()["pairs"][0]
        assert np.array_equal(a.forces(0), a.forces(1))
        assert a.result(0) == b.result(0)
        assert np.array_equal(a.forces(0), b.forces(0))
