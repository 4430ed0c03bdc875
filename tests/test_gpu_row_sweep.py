"""The sweep unrolled for each system's own slot count (spins in LDS, tables
in global memory: storage cap 1) against the general one (cap 0), bit for bit:
batches that mix 3, 4, 6 and 12 neighbours, FP32 and FP64, sizes around the
edges of a round of threads, with an onsite term and fields.  Both add a
field's terms in one order and draw the same numbers; the padding slots one of
them visits add exact zeros.  The FP64 tempering energies are summed by other
threads there and agree to 1e-12."""
import numpy as np
import pytest

import csmc
from csmc import workloads as W
from csmc.unitcell import addOnSite
from test_gpu_storage_modes import _ctx

pytestmark = pytest.mark.gpu


def _lattices(prec):
    on = W.honeycomb_kitaev(1.0, -2.0, h=[0.1, 0, 0.2])
    addOnSite(on, 1, np.diag([0.1, -0.2, 0.3]) + 0.05)
    cells = [(W.square_dm(-1.0, 0.1, (0.1, 0, 0.2)), (45, 46)), (W.triangular_dm(-0.9, -0.05, [0.3, 0.1, 0.0]), (33, 31)),
             (on, (19, 27)), (W.kgg_test_cell(), (32, 16)), (W.honeycomb_kitaev(1.0, -2.0), (1, 1)),
             (W.triangular_j1j2(1.0, 0.2), (13, 11)), (W.square_heisenberg(-1.0, (0, 0, 0.1)), (32, 64))]
    return [csmc.Lattice(shape, uc, 1.0, seed=k) for k, (uc, shape) in enumerate(cells)]


@pytest.mark.parametrize("which", ["mixed", "no_row_sweep"])
@pytest.mark.parametrize("prec", [32, 64])
def test_mixed_batch(prec, which):
    lats = _lattices(prec)
    if which == "no_row_sweep":  # slot counts that no sweep is unrolled for: the kernel without them
        lats = [lat for lat in lats if len(lat.unit_cell.bilinear) > (6 if prec == 32 else 4)]
        assert lats
    out = []
    for cap in (1, 0):
        print(f"[rows] {prec} {which} cap {cap}", flush=True)
        ctx = _ctx(cap)
        b = csmc.SpinBatch(lats, precision=prec, ctx=ctx)
        assert b.storage_mode() == cap
        b.randomize(3)
        b.set_counters(0)
        T, sg = np.linspace(0.2, 1.0, len(lats)), np.full(len(lats), 0.3)
        res = [np.asarray(b.sweep(csmc.OVERRELAX, n_sweeps=3)),
               np.asarray(b.sweep(csmc.METROPOLIS, T=T, n_sweeps=2, seed=5)),
               np.asarray(b.sweep(csmc.CONE_ADAPTIVE, T=T, sigma=sg, n_sweeps=2, seed=6)),
               np.asarray(b.anneal([0.8, 0.4], 7, 3, csmc.METROPOLIS, seed=7)), sg]
        out.append(res + [b.get_spins(r) for r in range(len(lats))])
        b.close()
        ctx.close()
    for x, y in zip(*out):
        assert np.array_equal(x, y)


@pytest.mark.parametrize("cell", ["kgg", "square_dm"])
def test_fp64_tempering(cell):
    uc = {"kgg": W.kgg_test_cell, "square_dm": lambda: W.square_dm(-1.0, 0.1, (0.1, 0, 0.2))}[cell]()
    lat, R, out = csmc.Lattice((17, 19), uc, 0.5, seed=1), 4, []
    for cap in (1, 0):
        ctx = _ctx(cap)
        b = csmc.SpinBatch([lat] * R, precision=64, ctx=ctx)
        assert b.storage_mode() == cap
        b.randomize(4)
        p = dict(t_thermalization=6, t_measurement=20, probe_rate=2, swap_rate=4, overrelaxation_rate=2,
                 report_interval=10 ** 9, checkpoint_rate=10 ** 9)
        b.pt_init(W.geometric_temperatures(0.3, 2.0, R), p, csmc.METROPOLIS, seed=9)
        b.pt_advance(-1)
        out.append((b.pt_state(), [b.get_spins(r) for r in range(R)]))
        b.close()
        ctx.close()
    (s1, x1), (s0, x0) = out
    for k in ("system_of_slot", "accepted_local", "accepted_exchange"):
        assert np.array_equal(s1[k], s0[k])
    assert np.allclose(s1["E"], s0["E"], rtol=1e-12, atol=1e-12)
    for x, y in zip(x1, x0):
        assert np.array_equal(x, y)
