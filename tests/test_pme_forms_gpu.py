"""The PME evaluation's forms against the FP64 oracle: transforms through planes and lines
(each line axis, prime lengths, the largest planes) and axis by axis, and x + d as the
difference from x (none displaced, displaced alike, displaced differently, exceptions
across) or in full (many displaced)."""
import ctypes

import numpy as np
import pytest

from atmmetaforce import _capi as C, pme
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


@pytest.mark.parametrize("n,chain", [(30, 0), (300, 140), (1700, 300), (3600, 0), (6000, 40)])
def test_direct_cells(gpu, n, chain):
    """Cells of 1 to 222 atoms (short and full chunks of 64, more than one staged batch of the
    neighbour cell) and exclusion groups longer than the staged rows of 128 atoms."""
    rng = np.random.default_rng(n)
    L = np.array([3.05, 3.1, 3.2])
    g = int(np.ceil(n ** (1 / 3)))
    lat = np.array([(i, j, k) for i in range(g) for j in range(g) for k in range(g)][:n], dtype=float)
    x = (lat + 0.5) * (L / g) + rng.uniform(-0.03, 0.03, (n, 3))
    q = rng.normal(0, 0.5, n)
    q -= q.mean()
    sig, eps = rng.uniform(0.15, 0.2, n), rng.uniform(0.1, 0.6, n)
    pairs = np.array([(i, i + 1) for i in range(5, 5 + chain)] + [(5, 5 + chain)] * (chain > 1)).reshape(-1, 2)
    zero = np.zeros(len(pairs))
    d = np.zeros((n, 3))
    # between lattice sites: the closest pairs at x + d stay below 1e7 kJ/mol/nm.  A shift off the lattice
    # (0.8, 0.9, 1.0) leaves a pair at 0.032 nm and 1.2e12 among 3600 atoms, past the 2^63 / 2^24 =
    # 5.5e11 that the forces' fixed-point sums hold.
    d[:max(1, n // 40)] = (L / g) * (2.5 if g > 4 else 0.5)
    print(f"[pme] {n} atoms, chain of {chain}", flush=True)
    with pme.ATMPMEForce(q, sig, eps, d, L, 1.0, exceptions=(pairs, zero, zero + 0.1, zero), params=PARAMS) as f:
        r, F, _ = f.evaluate(x)
    ref, Fref, p1, _ = _oracle_atm(x, q, sig, eps, L, pairs, zero, zero + 0.1, zero, d, PARAMS)
    # the sums' magnitudes (the self energy stands for the reciprocal sum, whose charges are rounded to 2^-36 e)
    scale = sum(abs(p1[k]) for k in ("direct_coulomb", "direct_lj", "exclusion_correction", "self"))
    assert abs(r["state1_energy"] - ref["U1"]) <= E_REL * max(1.0, scale)
    assert abs(r["energy"] - ref["W"]) <= E_REL * max(1.0, scale)
    assert np.abs(F - Fref).max() < F_ABS + 1e-12 * np.abs(Fref).max()


# an LJ pair passes the range of the fixed-point forces (5.5e11 kJ/mol/nm) below 0.05 nm
@pytest.mark.parametrize("dist", [0.05, 0.03, 0.01, 0.0])
@pytest.mark.parametrize("partner", ["stays", "displaced differently"])
def test_clash_at_x_leaves_the_other_state_alone(gpu, dist, partner):
    """A displaced atom on top of another at x, at the end of a leg where x + d is the physical
    state (direction -1, weight 0 for x): the energy and force of x + d are exact."""
    x, q, sig, eps, L, pairs, qq, es, ee, d = _small_system(seed=23)
    d[40:60] = (1.1, 1.2, 1.3)
    other = 200
    if partner != "stays":
        d[other] = (-0.55, 0.8, 0.3)
    x[50] = x[other] + dist * np.array([0.48, 0.6, 0.64])
    sig[[50, other]], eps[[50, other]] = 0.3, 0.5
    params = dict(PARAMS, lambda1=0.0, lambda2=0.0, alpha=0.0, w0=0.0, direction=-1.0)
    print(f"[pme] pair at {dist} nm, partner {partner}", flush=True)
    with pme.ATMPMEForce(q, sig, eps, d, L, 1.0, exceptions=(pairs, qq, es, ee), params=params) as f:
        r, F, _ = f.evaluate(x)
    U2, F2, p2 = po.nonbonded_pme(x + d, q, sig, eps, L, 1.0, pairs, qq, es, ee)
    # the sums' magnitudes (pairs of x + d may be close too), as the tests above
    scale = sum(abs(p2[k]) for k in ("direct_coulomb", "direct_lj", "exclusion_correction", "self"))
    assert abs(r["state2_energy"] - U2) <= E_REL * max(1.0, scale)
    if dist > 0.0:  # (two atoms in one place have no energy at x)
        U1, _, _ = po.nonbonded_pme(x, q, sig, eps, L, 1.0, pairs, qq, es, ee, forces=False)
        assert abs(r["state1_energy"] - U1) <= E_REL * abs(U1)
        assert abs(r["energy"] - U2) <= E_REL * max(1.0, scale)
        assert np.abs(F - F2).max() < F_ABS + 1e-12 * np.abs(F2).max()


def _set_particles(f, *arrays):
    C.check(f._lib.atm_pme_set_particles(f._h, *[np.ascontiguousarray(a, dtype=np.float64).ctypes.data_as(
        ctypes.POINTER(ctypes.c_double)) for a in arrays]))


def test_changed_particles_and_exceptions(gpu):
    """A change of the particles, displacements or exceptions gives the object new buffers, the one
    its forces are written to among them: what it computes next is what a new object computes."""
    x, q, sig, eps, L, pairs, qq, es, ee, d = _small_system(seed=29)
    rng = np.random.default_rng(5)
    kinds = (dict(), dict(state1_only=True), dict(forces=False))
    with pme.ATMPMEForce(q, sig, eps, d, L, 1.0, exceptions=(pairs, qq, es, ee), params=PARAMS) as f:
        for step in range(6):
            for kind in kinds:  # an evaluation of each kind captured before the change
                f.evaluate(x, **kind)
            d = np.where(rng.random((len(q), 1)) < 0.05 + 0.05 * (step % 2), rng.uniform(-1, 1, (len(q), 3)), 0.0)
            keep = rng.random(len(pairs)) < 0.8
            exc = (pairs[keep], qq[keep], es[keep], ee[keep])
            if step % 3 != 2:
                q = rng.permutation(q)
            _set_particles(f, q, sig, eps, d)
            f.set_exceptions(*exc)
            print(f"[pme] change {step}", flush=True)
            with pme.ATMPMEForce(q, sig, eps, d, L, 1.0, exceptions=exc, params=PARAMS) as new:
                for kind in kinds + kinds:
                    (r, F, p), (rn, Fn, pn) = f.evaluate(x, **kind), new.evaluate(x, **kind)
                    assert r == rn and (F is None or np.array_equal(F, Fn))
                    assert kind.get("state1_only") or p == pn


def test_far_positions(gpu):
    """Charged atoms at coordinates that no FP64 step brings back into the box: the evaluation ends
    inside its grids, and the next one is as it was."""
    x, q, sig, eps, L, pairs, qq, es, ee, d = _small_system(seed=31)
    far = x.copy()
    far[[7, 50, 399]] = [3e16, -1e17, 2e18], [-4e200, 1.0, 1e300], [2.0, -1e19, 1e25]  # atom 50 is displaced
    with pme.ATMPMEForce(q, sig, eps, d, L, 1.0, exceptions=(pairs, qq, es, ee), params=PARAMS) as f:
        r, F, _ = f.evaluate(x)
        for grid_state in (dict(), dict(state1_only=True)):
            print(f"[pme] far positions {grid_state}", flush=True)
            rf, Ff, _ = f.evaluate(far, **grid_state)
            assert np.isfinite(rf["state1_energy"]) and np.isfinite(Ff).all()
        r2, F2, _ = f.evaluate(x)
    assert r2 == r and np.array_equal(F2, F)


@pytest.mark.parametrize("classes", [1, 127, 128])
def test_displacement_classes(gpu, classes):
    """As many different displacements as the pairs of both states tell apart, and one more."""
    n = 2100
    rng = np.random.default_rng(classes)
    L = np.array([3.05, 3.1, 3.2])
    lat = np.array([(i, j, k) for i in range(13) for j in range(13) for k in range(13)][:n], dtype=float)
    x = (lat + 0.5) * (L / 13) + rng.uniform(-0.03, 0.03, (n, 3))
    q = rng.normal(0, 0.5, n)
    q -= q.mean()
    sig, eps = rng.uniform(0.15, 0.2, n), rng.uniform(0.1, 0.6, n)
    d = np.zeros((n, 3))
    at = rng.permutation(n)[:131]
    # between lattice sites, in whole steps of the lattice and a 1/512 of it that tells them apart
    d[at] = (L / 13) * (2.5 + rng.permutation(131)[:, None] % classes / 512.0)
    pairs = np.array([(at[0], at[1]), (at[0], 3), (4, 5)])
    zero = np.zeros(len(pairs))
    print(f"[pme] {classes} displacement classes", flush=True)
    with pme.ATMPMEForce(q, sig, eps, d, L, 1.0, exceptions=(pairs, zero, zero + 0.1, zero), params=PARAMS) as f:
        r, F, _ = f.evaluate(x)
    ref, Fref, p1, p2 = _oracle_atm(x, q, sig, eps, L, pairs, zero, zero + 0.1, zero, d, PARAMS)
    for key, want, p in (("state1_energy", ref["U1"], p1), ("state2_energy", ref["U2"], p2)):
        scale = sum(abs(p[k]) for k in ("direct_coulomb", "direct_lj", "exclusion_correction", "self"))
        assert abs(r[key] - want) <= E_REL * max(1.0, scale)
    assert np.abs(F - Fref).max() < F_ABS + 1e-12 * np.abs(Fref).max()
