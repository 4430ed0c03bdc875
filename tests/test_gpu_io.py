"""Spins and per-site evaluations between host and device: sizes around the
transfer kernels' 256-site blocks (odd ones end in a single double), and a
lattice of more sites than one staging block holds, and one either side of the
1 MB up to which uploads are staged, both precisions.  Results around and above
the size of a staging block."""
import numpy as np
import pytest

import csmc
from csmc import workloads as W
from conftest import random_spins

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [32, 64])
@pytest.mark.parametrize("shape", [(1, 1), (5, 51), (16, 16), (1, 257), (23, 45), (160, 273), (160, 274), (600, 601)])
def test_round_trip_and_site_energies(shape, prec):
    print(f"[io] {shape} {prec}", flush=True)
    lat = csmc.Lattice(shape, W.square_heisenberg(-1.0, (0.0, 0.0, 0.1)), 1.0, seed=1)
    N = lat.size
    rng = np.random.default_rng(3)
    b = csmc.SpinBatch([lat] * 2, precision=prec)
    s = [random_spins(N, 1.0, rng) for _ in range(2)]
    for i in range(2):
        b.set_spins(i, s[i])
    if prec == 32:
        s = [x.astype(np.float32).astype(np.float64) for x in s]
    h = np.array([0.0, 0.0, 0.1])
    for i in range(2):
        assert np.array_equal(b.get_spins(i), s[i])
        # F = -(sum of the four neighbours), H = F - h, e = s.F - s.h; each a
        # sum of at most 18 products of size 1
        g = s[i].reshape(*shape, 3)
        F = -sum(np.roll(g, d, a) for a in (0, 1) for d in (1, -1)).reshape(N, 3)
        assert np.max(np.abs(b.local_field(i) - (F - h))) <= 20 * 2.0 ** -52 * 4
        assert np.max(np.abs(b.site_energy(i) - np.sum(s[i] * (F - h), axis=1))) <= 20 * 2.0 ** -52 * 4
    b.close()


@pytest.mark.parametrize("n_temps", [1023, 1024])
def test_accepted_counts_around_a_staging_block(n_temps):
    """1024 systems and 1023 temperatures fill a block of 8 MB with the
    temperatures and the flag, one more does not fit: the counts are those of
    the same annealing in two calls"""
    lat = csmc.Lattice((2, 3), W.square_heisenberg(-1.0, (0.0, 0.0, 0.1)), 1.0, seed=1)
    T = np.linspace(2.0, 0.5, n_temps)
    got = []
    for cuts in ([0, n_temps], [0, 500, n_temps]):
        b = csmc.SpinBatch([lat] * 1024, precision=64)
        b.randomize(3)
        acc = [b.anneal(T[i:j], 3, 0, csmc.METROPOLIS, seed=5) for i, j in zip(cuts, cuts[1:])]
        got.append((np.concatenate(acc, axis=1), [b.get_spins(i) for i in (0, 511, 1023)]))
        b.close()
    assert np.array_equal(got[0][0], got[1][0]) and 0 < got[0][0].mean() < 12
    for x, y in zip(got[0][1], got[1][1]):
        assert np.array_equal(x, y)


def test_gradients_larger_than_a_staging_block():
    """gradients that leave in several ranges: those of the same systems in a
    batch of their own"""
    lat = csmc.Lattice((4, 3, 5), W.pyrochlore_mixed(), 1.0, seed=1)
    nl = lat.unit_cell.n_params()
    n = (9 << 20) // (8 * nl) + 3
    rng = np.random.default_rng(8)
    some = [0, 1, n // 2, n - 2, n - 1]
    s = {i: random_spins(lat.size, 1.0, rng) for i in some}
    b, few = csmc.SpinBatch([lat] * n, precision=64), csmc.SpinBatch([lat] * len(some), precision=64)
    b.randomize(4)
    for k, i in enumerate(some):
        b.set_spins(i, s[i])
        few.set_spins(k, s[i])
    for _ in range(2):
        J, j, S, x = b.grad_couplings(), few.grad_couplings(), b.grad_spins(), few.grad_spins()
        for k, i in enumerate(some):
            assert np.array_equal(J[i], j[k]) and np.array_equal(S[i], x[k])
        few.total_energy()
    b.close()
    few.close()


@pytest.mark.parametrize("R", [1638, 1639])
def test_observables_around_a_staging_block(R):
    """the binned sums of 1638 slots fill a block of 8 MB, one more slot is a
    second range: after a single probe every slot's mean energy is its energy"""
    lat = csmc.Lattice((2, 3), W.square_heisenberg(-1.0, (0.0, 0.0, 0.1)), 1.0, seed=1)
    b = csmc.SpinBatch([lat] * R, precision=64)
    b.randomize(3)
    p = dict(t_thermalization=4, t_measurement=1, probe_rate=4, swap_rate=10 ** 6, overrelaxation_rate=1,
             report_interval=10 ** 9, checkpoint_rate=10 ** 9)
    b.pt_init(np.geomspace(0.1, 2.0, R), p, csmc.METROPOLIS, seed=9)
    b.pt_advance(-1)
    E = b.pt_state()["E"]
    assert np.array_equal(b.pt_observables()["energy"], E) and len(set(E)) > R // 2
    b.close()


def test_contexts_share_the_staging_blocks():
    """more contexts than blocks kept, opened and closed in turn, each with
    transfers of another size"""
    uc = W.square_heisenberg(-1.0, (0.0, 0.0, 0.1))
    rng = np.random.default_rng(4)
    for k in range(12):
        ctxs = [csmc.Context() for _ in range(1 + k % 3)]
        for j, ctx in enumerate(ctxs):
            lat = csmc.Lattice((8 + 40 * j, 9), uc, 1.0, seed=1)
            b = csmc.SpinBatch([lat], precision=64, ctx=ctx)
            s = random_spins(lat.size, 1.0, rng)
            b.set_spins(0, s)
            assert np.array_equal(b.get_spins(0), s)
        for ctx in ctxs:
            ctx.close()
