"""Host positions, parameters and device parameters on their way in and forces on their way
out through page-locked memory: whole values, so the results of both routes are the same."""
import numpy as np
import pytest
import torch

from atmmetaforce import ATMBatch, workloads as W

pytestmark = pytest.mark.gpu


def _systems(sizes):
    p = W.ATMParams(0.2, 0.4, 0.1, 110.0, 0.0, 200.0, 100.0, 0.0625, 1.0)
    L = 3.0
    return [W.lattice_system(n, L, 0.9, max(1, n // 50), (L / 4, L / 4, L / 4), 7 + n, p) for n in sizes]


# one atom, odd tails of the 16-byte rows, the edges of the 256-atom blocks
@pytest.mark.parametrize("sizes", [(1,), (3, 255, 2), (256, 257, 1023, 64, 511)])
def test_positions_and_forces(gpu, sizes):
    systems = _systems(sizes)
    rng = np.random.default_rng(len(sizes))
    with ATMBatch(systems) as b:
        for step in range(3):  # the uploads run on while the next system's positions are converted
            xs = [(s.positions + rng.uniform(-0.02, 0.02, s.positions.shape)).astype(np.float32) for s in systems]
            for k, x in enumerate(xs):
                b.set_positions(k, x + 100.0)  # overwritten before anything reads it
                b.set_positions(k, x)
                b.set_params(k, (0.1 * step, 0.5, 0.1, 110.0, 0.0, 200.0, 100.0, 0.0625, 1.0))
            b.compute()
            host = [(b.result(k), b.forces(k), b.forces_fixed(k)) for k in range(len(sizes))]
            dev = torch.as_tensor(np.concatenate(xs), device="cuda")
            torch.cuda.synchronize()
            b.set_positions_device(dev.data_ptr())
            b.compute()
            for k in list(range(len(sizes))) * 2:  # one after the other, and again from the first
                r, F, fix = host[k]
                assert b.result(k) == r
                assert np.array_equal(b.forces(k), F)
                assert np.array_equal(np.rint(F * 2.0 ** 24).astype(np.int64), fix)
            b.clear_forces()  # the systems sent ahead of being asked for are not shown after it
            order = list(range(len(sizes))) + [0]
            assert all(not b.forces(k).any() for k in order)
            b.compute()
            for k in order + order[::-1] + order:
                assert np.array_equal(b.forces(k), host[k][1])
            b.compute(plain=True)  # records of the host-side path beside those of the batched one
            assert b.result(0)["state1_energy"] == pytest.approx(host[0][0]["state1_energy"], rel=1e-12, abs=1e-9)


def test_device_parameters_refused_unchanged(gpu):
    systems = _systems((255, 700))
    n = 955
    with ATMBatch(systems) as b:
        b.compute()
        before = [b.result(k) for k in range(2)], b.forces(1)
        cols = [torch.as_tensor(np.concatenate([getattr(s, c) for s in systems]) * 0.9, device="cuda", dtype=torch.float64)
                for c in ("charges", "sigmas", "epsilons")]
        cols[1][n - 1] = -1.0
        torch.cuda.synchronize()
        with pytest.raises(Exception, match="1 atoms with a non-finite parameter"):
            b.set_particles_device(*[c.data_ptr() for c in cols])
        b.compute()
        assert [b.result(k) for k in range(2)] == before[0] and np.array_equal(b.forces(1), before[1])


def test_reads_leave_the_stream_idle(gpu):
    """A force read returns with its work done: nothing of another system is still on its way on
    the caller's stream."""
    systems = _systems((40000, 30001, 40000, 39999, 7, 40000, 20000))
    stream = torch.cuda.Stream()
    with ATMBatch(systems) as b:
        b.set_stream(stream.cuda_stream)
        b.compute()
        first = []
        for k in range(len(systems)):
            first.append(b.forces(k))
            assert stream.query(), k
        for k in (3, 4, 0, 1, 6, 5, 2):
            assert np.array_equal(b.forces(k), first[k])
            assert stream.query(), k
        b.set_stream(None)


def test_systems_beyond_the_staging(gpu):
    """Positions of more than 65,536 atoms go in pieces, forces of more than 174,762 come in pieces,
    and reads one after the other send what fits."""
    p = W.ATMParams(0.2, 0.4, 0.1, 110.0, 0.0, 200.0, 100.0, 0.0625, 1.0)
    systems = [W.lattice_system(n, (n / 33.75) ** (1.0 / 3.0), 0.6, 20, (1.0, 1.0, 1.0), 3 + n, p)
               for n in (65536, 180001, 65537, 60000, 131075)]
    rng = np.random.default_rng(2)
    xs = [(s.positions + rng.uniform(-0.02, 0.02, s.positions.shape)).astype(np.float32) for s in systems]
    with ATMBatch(systems) as b:
        for k, x in enumerate(xs):
            b.set_positions(k, x)
        b.compute()
        order = list(range(len(xs))) + [3, 4, 0, 1, 2, 2]
        host = [(b.result(k), b.forces(k)) for k in order]
        dev = torch.as_tensor(np.concatenate(xs), device="cuda")
        torch.cuda.synchronize()
        b.set_positions_device(dev.data_ptr())
        b.compute()
        for k, (r, F) in zip(order, host):
            assert b.result(k) == r
            fixed = b.forces_fixed(k)
            assert np.array_equal(np.rint(F * 2.0 ** 24).astype(np.int64), fixed)
            assert np.abs(F).max() > 1.0
