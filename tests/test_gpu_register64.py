"""The FP64 register-table sweep kernel against the LDS-array kernel (the
storage cap selects it), bit for bit: spins, acceptance, energies and
tempering state.  Both visit the same sites with the same threads, add a
field's terms in the same order and draw the same numbers, so no tolerance is
needed.  Layouts at the edges of the kernel's 512-site slots and of its
dispatch (3 or 4 neighbours, at most 8 slots and 4 colours; more systems than
CUs)."""
import numpy as np
import pytest

import csmc
from csmc import workloads as W
from csmc.unitcell import addOnSite
from test_gpu_storage_modes import _ctx

pytestmark = pytest.mark.gpu


def _onsite(uc):
    addOnSite(uc, 1, np.diag([0.1, -0.2, 0.3]) + 0.05)
    return uc


LAYOUTS = [  # (name, unit cell, shape, S)
    ("one_wave", lambda: W.square_heisenberg(-1.0, (0, 0.2, 0.1)), (10, 10), 1.0),
    ("one_cell", lambda: W.honeycomb_kitaev(1.0, -2.0), (1, 1), 0.5),
    ("full_slot", lambda: W.honeycomb_kitaev(1.0, -2.0, h=[0.1, 0, 0.2]), (16, 32), 0.5),
    ("over_a_slot", lambda: _onsite(W.honeycomb_kitaev(1.0, -2.0)), (19, 27), 0.5),  # 513 sites a run
    ("full_matrices", W.kgg_test_cell, (24, 24), 0.5),
    ("full_matrices_4", lambda: W.square_dm(-1.0, 0.1, (0.1, 0, 0.2)), (30, 36), 1.0),
    ("three_colours", lambda: W.square_dm(-1.0, 0.1, (0.1, 0, 0.2)), (45, 45), 1.0),
    ("eight_slots", lambda: W.square_heisenberg(-1.0, (0, 0, 0)), (64, 64), 1.0),
    ("nine_slots", lambda: W.square_heisenberg(-1.0, (0, 0, 0)), (64, 66), 1.0),  # the other kernel
]


# more systems than a device has CUs: workgroups of 4 waves at most stay with the
# kernel, of larger ones only some of the calls
QUEUED = [
    ("queued_four_waves", lambda: W.square_heisenberg(-1.0, (0, 0.2, 0.1)), (16, 32), 1.0),
    ("queued_five_waves", lambda: W.square_heisenberg(-1.0, (0, 0.2, 0.1)), (20, 32), 1.0),
    ("queued_full_matrices", lambda: W.square_dm(-1.0, 0.1, (0.1, 0, 0.2)), (20, 27), 1.0),
    ("queued_six_neighbours", lambda: W.triangular_dm(-1.0, 0.1, (0.1, 0, 0.2)), (30, 30), 1.0),  # the other kernel
]


@pytest.mark.parametrize("case", LAYOUTS + QUEUED, ids=[c[0] for c in LAYOUTS + QUEUED])
def test_same_bits_as_lds_arrays(case):
    name, mk, shape, S = case
    print(f"[register64] {name}", flush=True)
    R = 300 if case in QUEUED else 3
    # the calls that run in the kernel: overrelaxation, Metropolis, annealing, tempering
    runs = {"nine_slots": "----", "queued_six_neighbours": "----", "queued_five_waves": "o-a-",
            "queued_full_matrices": "o---"}.get(name, "omat")
    lats = [csmc.Lattice(shape, mk(), S, seed=1)] * R
    out = []
    for cap in (3, 2):
        ctx = _ctx(cap)
        b = csmc.SpinBatch(lats, precision=64, ctx=ctx)
        b.randomize(11)
        b.set_counters(0)
        T, sg = np.resize([0.2, 0.5, 1.0], R), np.full(R, 0.3)

        def ran(call, result=None):  # the call was made by the expected kernel
            form, parts = b.last_form()
            assert parts == 1 and (form == 4) == (cap == 3 and call in runs), (call, form)
            return np.asarray(result)

        res = [ran("o", b.sweep(csmc.OVERRELAX, n_sweeps=3)),
               ran("m", b.sweep(csmc.METROPOLIS, T=T, n_sweeps=2, seed=5)),
               ran("m", b.sweep(csmc.CONE_ADAPTIVE, T=T, sigma=sg, n_sweeps=2, seed=6)),
               ran("o", b.sweep(csmc.DETERMINISTIC, n_sweeps=1)),
               ran("a", b.anneal([0.8, 0.4], 5, 2, csmc.METROPOLIS, seed=7)), sg]
        res += [b.get_spins(r) for r in range(R)]
        p = dict(t_thermalization=6, t_measurement=20, probe_rate=2, swap_rate=4, overrelaxation_rate=2,
                 report_interval=10 ** 9, checkpoint_rate=10 ** 9)
        b.pt_init(W.geometric_temperatures(0.3, 2.0, R), p, csmc.METROPOLIS, seed=9)
        b.pt_advance(-1)
        ran("t")
        st = b.pt_state()
        res += [np.asarray(st[k]) for k in ("system_of_slot", "accepted_local", "accepted_exchange", "E")]
        res += [b.get_spins(r) for r in range(R)]
        out.append(res)
        b.close()
        ctx.close()
    for x, y in zip(*out):
        assert np.array_equal(x, y)
