"""Calls that make captured evaluations over while one of them may still be running: the next
results are those of a context that waited in between."""
import numpy as np
import pytest

from atmmetaforce import ATMBatch, workloads as W

pytestmark = pytest.mark.gpu


def _systems():
    p = W.ATMParams(0.2, 0.4, 0.1, 110.0, 0.0, 200.0, 100.0, 0.0625, 1.0)
    base = W.lattice_system(9001, 6.5, 0.9, 40, (1.6, 1.6, 1.6), 17, p)
    return W.replica_batch(6, base=base)


def _exceptions(b, systems):
    for k, s in enumerate(systems):
        at = np.arange(0, 3000, 3)
        b.set_exceptions(k, np.stack([at, at + 1], 1), np.zeros(len(at)), np.full(len(at), 0.1), np.zeros(len(at)))


@pytest.mark.parametrize("change", ["exceptions", "gradients", "tuning"])
def test_change_after_an_evaluation_that_was_not_waited_for(gpu, change):
    systems = _systems()
    seen = []
    for wait in (True, False):
        with ATMBatch(systems) as b:
            b.compute()
            print(f"[graphs] {change}, wait {wait}", flush=True)
            for _ in range(8):
                b.evaluate()
            if wait:
                b.synchronize()
            if change == "exceptions":
                _exceptions(b, systems)
            elif change == "gradients":
                b.compute(forces=False, param_grads=True)
            else:
                b.set_tuning(1.15, 2, 2)
            b.compute()
            seen.append(([b.result(k) for k in range(6)], [b.forces(k) for k in range(6)]))
    assert seen[0][0] == seen[1][0]
    assert all(np.array_equal(x, y) for x, y in zip(seen[0][1], seen[1][1]))
