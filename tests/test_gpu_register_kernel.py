"""The register-table sweep kernel over the layouts its dispatch tells apart,
against the LDS-array kernel bit for bit, and the chained exchange schedule
with probes before, at and after an exchange and with exchanges whose indices
are 1 to 8 apart, against one launch per period.  The bodies are those of test_gpu_storage_modes and
test_gpu_pt_chain."""
import numpy as np
import pytest

import csmc
from csmc import workloads as W
from csmc.unitcell import addOnSite
from test_gpu_pt_chain import test_chained_pt_matches_per_period_launches as chain_body
from test_gpu_storage_modes import _ctx, test_register_mode_matches_lds_mode as modes_body

pytestmark = pytest.mark.gpu


def _onsite(uc):
    addOnSite(uc, 1, np.diag([0.1, -0.2, 0.3]) + 0.05)
    return uc


LAYOUTS = [  # (name, unit cell, shape, S, expected modes (cap 3, cap 2))
    # two full colours of 2 and of 4 slots, without and with a field or onsite term
    ("two_colour_2_plain", lambda: W.square_heisenberg(-1.0, (0, 0, 0)), (64, 64), 1.0, (3, 2)),
    ("two_colour_2_field", lambda: W.square_heisenberg(-1.0, (0, 0.2, 0.1)), (64, 64), 1.0, (3, 2)),
    ("two_colour_4_field", lambda: W.honeycomb_kitaev(1.0, -2.0, h=[0.1, 0, 0.2]), (64, 64), 0.5, (3, 2)),
    ("two_colour_2_onsite", lambda: _onsite(W.square_heisenberg(-1.0, (0, 0, 0))), (64, 64), 1.0, (3, 2)),
    # one colour short of a slot, one site over a slot, a slot shared by few
    ("two_colour_short", lambda: W.honeycomb_kitaev(1.0, -2.0), (63, 65), 0.5, (3, 2)),
    ("over_a_slot", lambda: W.honeycomb_kitaev(1.0, -2.0), (25, 41), 0.5, (3, 2)),
    ("three_colours", lambda: W.square_dm(-1.0, 0.1, (0.1, 0, 0.2)), (45, 45), 1.0, (3, 2)),
    ("six_neighbours", lambda: W.triangular_dm(-0.9, -0.05, [0.3, 0.1, 0.0]), (30, 33), 1.0, (3, 2)),
    ("six_neighbours_six_slots", lambda: W.triangular_dm(-0.9, -0.05, [0.3, 0.1, 0.0]), (57, 60), 1.0, (3, 2)),
    ("one_cell", lambda: W.honeycomb_kitaev(1.0, -2.0), (1, 1), 0.5, (3, 2)),
]


@pytest.mark.parametrize("case", LAYOUTS, ids=[c[0] for c in LAYOUTS])
def test_layouts(case):
    print(f"[register] {case[0]}", flush=True)
    modes_body(case)


def _schedule(probe, swap, orr, t_th=7, t_meas=90):
    return dict(t_thermalization=t_th, t_measurement=t_meas, probe_rate=probe, swap_rate=swap, overrelaxation_rate=orr,
                report_interval=10 ** 9, checkpoint_rate=10 ** 9)


SCHEDULES = [
    ("every_probe", _schedule(1, 6, 3)),       # several probes before an exchange is resolved
    ("no_overrelaxation", _schedule(2, 3, 0)),  # a Metropolis sweep follows every exchange
    ("coprime", _schedule(7, 5, 5)),
    ("sparse_exchange", _schedule(4, 12, 2, t_th=0)),
    # consecutive exchanges eight indices apart, the length of the record ring
    ("apart_8_1", _schedule(5, 1, 8, t_meas=400)),
    ("apart_16_2", _schedule(16, 2, 16, t_meas=800)),
]


@pytest.mark.parametrize("prec", [32, 64])
@pytest.mark.parametrize("sched", SCHEDULES, ids=[s[0] for s in SCHEDULES])
def test_schedules(sched, prec):
    print(f"[register] {sched[0]} {prec}", flush=True)
    chain_body((sched[0], lambda: W.kgg_test_cell(), (6, 5), 0.5, prec, 5, csmc.CONE_ADAPTIVE, sched[1]))


@pytest.mark.parametrize("cell", ["dm", "diagonal"])
def test_six_slots_keep_energies(cell):
    """six neighbours with five or six slots: the same terms in the same order
    as the LDS arrays, so equal FP64 energies"""
    J = (-0.05, [0.3, 0.1, 0.0]) if cell == "dm" else (0.0, [0.0, 0.0, 0.0])
    lat = csmc.Lattice((60, 54), W.triangular_dm(-0.9, *J), 1.0, seed=1)
    out = []
    for cap in (3, 2):
        ctx = _ctx(cap)
        b = csmc.SpinBatch([lat] * 3, precision=32, ctx=ctx)
        assert b.storage_mode() == cap
        b.randomize(5)
        b.pt_init(W.geometric_temperatures(0.3, 2.0, 3), _schedule(2, 4, 2), csmc.METROPOLIS, seed=9)
        b.pt_advance(-1)
        out.append((b.pt_state()["E"], [b.get_spins(r) for r in range(3)]))
        b.close()
        ctx.close()
    assert np.array_equal(out[0][0], out[1][0])
    for x, y in zip(out[0][1], out[1][1]):
        assert np.array_equal(x, y)
