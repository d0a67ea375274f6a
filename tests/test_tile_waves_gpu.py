"""The tile kernel's waves per group (2, 4, 8 or 16, from the number of groups): lists
shorter than the waves that share them, each block size, and the sizes where the choice
changes, against the FP64 oracle."""
import numpy as np
import pytest

from atmmetaforce import ATMBatch, workloads as W
from oracle import oracle

pytestmark = pytest.mark.gpu

RHO = 23000.0 / 8.8 ** 3


def _systems(count, n, cutoff=0.9):
    L = max((n / RHO) ** (1.0 / 3.0), 2.0 * cutoff + 0.05)
    p = W.ATMParams(0.2, 0.4, 0.1, 110.0, 0.0, 200.0, 100.0, 0.0625, 1.0)
    base = W.lattice_system(n, L, cutoff, max(1, n // 50), (L / 4, L / 4, L / 4), 31 + n, p)
    return W.replica_batch(count, base=base) if count > 1 else [base]


# one group with fewer entries than waves; 16 waves; 16 -> 8 (256 groups); 8 -> 4 (1,280);
# 4 -> 2 (5,120)
@pytest.mark.parametrize("count,n", [(1, 7), (1, 65), (3, 1001), (5, 2501), (6, 2501), (8, 9001), (22, 9001), (24, 12007)])
def test_waves_per_group(gpu, count, n):
    systems = _systems(count, n)
    with ATMBatch(systems) as b:
        b.compute()
        counts = b.list_stats()["pairs"]
        for k in sorted({0, count // 2, count - 1}):
            s = systems[k]
            ref, Fref = oracle.atm_eval(s)
            r = b.result(k)
            # FP64 pair energies in another order: 1e-13 of the sum of their magnitudes
            assert abs(r["state1_energy"] - ref["U1"]) <= 1e-13 * max(ref["abs1"], 1.0)
            assert counts[2 * k] == len(oracle.pairs(s.positions, s.box, s.cutoff))
            # FP32 force vectors (2^-24 each) and per-lane sums of up to ~100 of them
            assert np.linalg.norm(b.forces(k) - Fref) <= 1e-6 * max(np.linalg.norm(Fref), 1e-3)
        e = b.results()
        b.compute(forces=False)
        assert [r["energy"] for r in b.results()] == pytest.approx([r["energy"] for r in e], rel=1e-12)
