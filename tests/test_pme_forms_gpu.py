"""The PME evaluation's forms against the FP64 oracle: transforms through planes and lines
(each line axis, prime lengths, the largest planes) and axis by axis, and x + d as the
difference from x (none displaced, displaced alike, displaced differently, exceptions
across) or in full (many displaced)."""
import numpy as np
import pytest

from atmmetaforce import pme
from oracle import pme_oracle as po
from test_pme_gpu import E_REL, F_ABS, PARAMS, _oracle_atm, _small_system

pytestmark = pytest.mark.gpu


def _displacements(form, n):
    d = np.zeros((n, 3))
    if form == "alike":
        d[40:60] = (1.1, 1.2, 1.3)
    elif form == "mixed":
        # atoms 3, 4 have exceptions with atoms that stay; 31 and 32 are excepted from each other
        for k, i in enumerate((3, 4, 31, 32, 50, 51)):
            d[i] = (0.7 + 0.1 * k, -0.4, 0.3 * (k % 2))
    elif form == "many":
        d[100:300] = (0.9, 0.0, -1.2)
    return d


@pytest.mark.parametrize("form,grid", [("none", None), ("alike", None), ("mixed", None), ("many", None),
                                       ("alike", (11, 13, 17)), ("alike", (100, 12, 9)), ("mixed", (9, 100, 12)),
                                       ("many", (12, 9, 100)), ("alike", (60, 64, 72)), ("mixed", (72, 72, 75))])
def test_forms(gpu, form, grid):
    x, q, sig, eps, L, pairs, qq, es, ee, _ = _small_system(seed=21)
    d = _displacements(form, len(q))
    print(f"[pme] {form} grid {grid}", flush=True)
    with pme.ATMPMEForce(q, sig, eps, d, L, 1.0, exceptions=(pairs, qq, es, ee), params=PARAMS, grid=grid) as f:
        r, F, parts = f.evaluate(x)
        r1, F1, _ = f.evaluate(x, state1_only=True)
        r2, F2, parts2 = f.evaluate(x)
    assert r2 == r and np.array_equal(F2, F) and parts2 == parts
    ref, Fref, p1, p2 = _oracle_atm(x, q, sig, eps, L, pairs, qq, es, ee, d, PARAMS, grid=grid)
    for got, want in ((r["state1_energy"], ref["U1"]), (r["state2_energy"], ref["U2"]), (r["energy"], ref["W"]),
                      (r1["state1_energy"], ref["U1"])):
        assert abs(got - want) <= E_REL * max(1.0, abs(want)), (got, want)
    for s, p in ((1, p1), (2, p2)):
        assert abs(parts[f"direct{s}"] - (p["direct_coulomb"] + p["direct_lj"])) < 1e-8 * abs(p["direct_coulomb"])
        assert abs(parts[f"reciprocal{s}"] - p["reciprocal"]) < 1e-8 * abs(p["reciprocal"])
    # clashes at x + d leave forces of up to 1e9 in one state: relative where it is larger
    assert np.all(np.abs(F - Fref) < F_ABS + 1e-12 * np.abs(Fref).max())
    assert np.abs(F1 - po.nonbonded_pme(x, q, sig, eps, L, 1.0, pairs, qq, es, ee, grid=grid)[1]).max() < F_ABS
