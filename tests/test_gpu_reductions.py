"""Sums over the sites of a system that several workgroups or many threads
share: total energy and magnetisation around the sizes where a system is cut
into ranges, alone and in an uneven batch, and coupling gradients with every
kind of term.

Bounds: every sum has at most a few hundred additions in sequence per thread
and in the ranges after it, so its rounding error is below 1e3 x 2^-53 < 1.2e-13
times the sum of the absolute values of its terms."""
import numpy as np
import pytest

import csmc
import oracle.oracle as orc
from csmc import workloads as W
from conftest import random_spins
from test_gpu_adjoint import _random_cell

pytestmark = pytest.mark.gpu
REL = 1.2e-13


def _magnitude(uc, N, S):
    """a bound of the sum of the absolute values of the energy's terms: every
    coupling entry times one product of spin components per cell and role"""
    n = 0.0
    for q, terms in ((1, uc.field), (2, uc.onsite), (2, uc.bilinear), (3, uc.cubic), (4, uc.quartic)):
        for t in terms:
            M = next(x for x in reversed(t) if isinstance(x, np.ndarray) and x.dtype == np.float64)
            n += np.abs(M).sum() * S ** q
    return n * N


# side lengths around one range (1024 sites) and with a last range of one site
@pytest.mark.parametrize("prec", [32, 64])
@pytest.mark.parametrize("cell,shape", [("square", (1, 1)), ("square", (31, 33)), ("square", (32, 32)),
                                        ("square", (25, 41)), ("square", (45, 45)), ("honeycomb", (40, 37)),
                                        ("pyrochlore", (7, 7, 7))])
def test_energy_and_magnetisation(cell, shape, prec):
    print(f"[reductions] {cell} {shape} {prec}", flush=True)
    uc = {"square": W.square_heisenberg, "honeycomb": W.kgg_test_cell, "pyrochlore": W.pyrochlore_mixed}[cell]()
    lat = csmc.Lattice(shape, uc, 1.0, seed=2)
    T = orc.Tables(uc, shape)
    rng = np.random.default_rng(5)
    b = csmc.SpinBatch([lat] * 3, precision=prec)
    spins = [random_spins(lat.size, 1.0, rng) for _ in range(3)]
    for i in range(3):
        b.set_spins(i, spins[i])
    if prec == 32:
        spins = [s.astype(np.float32).astype(np.float64) for s in spins]
    E, parts = b.total_energy(parts=True)
    M = b.magnetization()
    for i in range(3):
        e, p = orc.total_energy(T, spins[i], parts=True)
        tol = REL * _magnitude(uc, 12 * lat.size, 1.0)
        assert abs(E[i] - e) <= tol, (cell, shape, i)
        assert np.max(np.abs(parts[i] - np.asarray(p))) <= 4 * tol
        assert np.max(np.abs(M[i] - spins[i].sum(axis=0))) <= REL * lat.size
    b.close()


@pytest.mark.parametrize("prec", [32, 64])
def test_uneven_batch(prec):
    """lattices of one and of several ranges in one batch, the large ones
    first, last and between"""
    uc = W.square_heisenberg()
    shapes = [(33, 64), (1, 1), (3, 3), (41, 25), (2, 5), (32, 32), (5, 5), (64, 65)]
    lats = [csmc.Lattice(s, uc, 1.0, seed=2) for s in shapes]
    rng = np.random.default_rng(6)
    b = csmc.SpinBatch(lats, precision=prec)
    spins = [random_spins(lat.size, 1.0, rng) for lat in lats]
    for i, s in enumerate(spins):
        b.set_spins(i, s)
    if prec == 32:
        spins = [s.astype(np.float32).astype(np.float64) for s in spins]
    E, parts = b.total_energy(parts=True)
    M = b.magnetization()
    for i, shape in enumerate(shapes):
        e, p = orc.total_energy(orc.Tables(uc, shape), spins[i], parts=True)
        tol = REL * _magnitude(uc, 12 * lats[i].size, 1.0)
        assert abs(E[i] - e) <= tol, shape
        assert np.max(np.abs(parts[i] - np.asarray(p))) <= 4 * tol, shape
        assert np.max(np.abs(M[i] - spins[i].sum(axis=0))) <= REL * lats[i].size, shape
    b.close()


@pytest.mark.parametrize("name,mk,shape,bc", [
    ("triangular", W.triangular_j1j2, (33, 17), "periodic"),    # groups of terms, one basis
    ("kgg_open", W.kgg_test_cell, (23, 24), "open"),            # reversed roles, absent partners, fields
    ("pyrochlore", W.pyrochlore_mixed, (3, 4, 5), "periodic"),  # cubic, quartic, onsite
    ("patterns", W.tensor_pattern_cell, (9, 5), "periodic"),    # repeated bases, dense tensors
    ("random", _random_cell, (5, 4), "open"),
    ("one_site", W.square_heisenberg, (1, 1), "open"),
    ("short_run", W.square_heisenberg, (8, 17), "periodic"),     # a wave and a bit
    ("long_run", W.kgg_test_cell, (33, 40), "periodic"),         # more sites than a workgroup has threads
])
def test_energy_is_linear_in_the_couplings(name, mk, shape, bc):
    """total_energy is linear in the couplings, so it equals the couplings
    times their gradient; and a coupling's gradient is the energy of the cell
    with that coupling at 1 and the others at nothing"""
    print(f"[reductions] couplings {name}", flush=True)
    uc = mk()
    lat = csmc.Lattice(shape, uc, 1.0, bc=bc, seed=3)
    T = orc.Tables(uc, shape, periodic=bc == "periodic")
    rng = np.random.default_rng(7)
    b = csmc.SpinBatch([lat] * 2, precision=64)
    spins = [random_spins(lat.size, 1.0, rng) for _ in range(2)]
    for i in range(2):
        b.set_spins(i, spins[i])
    G = b.grad_couplings()
    assert np.array_equal(G, b.grad_couplings())  # the sums' order is fixed
    p = uc.params()
    tol = REL * _magnitude(uc, 12 * lat.size, 1.0)
    for i in range(2):
        assert abs(G[i] @ p - orc.total_energy(T, spins[i])) <= tol, (name, i)
    for k in rng.choice(len(p), size=min(len(p), 24), replace=False):
        theta = np.where(p != 0, 1e-300, 0.0)  # keep every term of the cell, at no weight
        theta[k] = 1.0
        Tk = orc.Tables(uc.with_params(theta), shape, periodic=bc == "periodic")
        assert abs(G[0][k] - orc.total_energy(Tk, spins[0])) <= REL * 12 * lat.size, (name, k)
    b.close()
