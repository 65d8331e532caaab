"""The forms of the step kernels give the same records, bit for bit: one lane per trajectory over the slots in place
(what a replayed graph runs), four lanes per trajectory (runs of at most 16384 trajectories), and the running
slots packed into full waves while a larger run drains, first with one lane, then with four; including
attempts that end in a field error and launches that stop anywhere in the random stream."""
import numpy as np
import pytest
import feature_setups as fs

from spectrum_amd import cartesian
from spectrum_amd import configs as cf
from spectrum_amd import engine as E

pytestmark = pytest.mark.gpu

MANY = 16640   # a block of slots beyond the largest run of the four-lane form: its drain is packed


def wide_grid():
    return cartesian.parker_spiral(12, 100.0)


def small_grid():
    """A grid that most trajectories leave: field errors, retries and abandoned trajectories."""
    return cartesian.parker_spiral(6, 6.0)


SETUPS = {
    "modulation": lambda: cf.parker_modulation(n_energies=7, r_start_au=20.0, t_limit_years=8.0 / 365.0, time_action=0),
    "modulation_tilted": lambda: cf.parker_modulation(n_energies=7, r_start_au=20.0, t_limit_years=3.0 / 365.0, time_action=0,
                                                      sw=cf.solarwind(axis=(0.0, 0.6, 0.8))),
    "radial": lambda: cf.parker_modulation_radial(n_energies=3, inner_au=0.8, outer_au=3.0),
    "shock_source": lambda: cf.dsa_shock(t_limit_days=0.005, src_ratio=1.01),
    "guiding": lambda: cf.gc_diff_scatt(t_limit_days=0.03),
    "guiding_uniform": lambda: cf.gc_uniform(t_limit=40.0),
    "uniform": lambda: cf.uniform_walk(t_limit=300.0),
    "grid": lambda: cf.parker_modulation_cartesian(wide_grid(), t_limit_years=2.0 / 365.0),
    "grid_anisotropic": lambda: cf.parker_modulation_cartesian(wide_grid(), kap_rat=0.3, t_limit_years=2.0 / 365.0),
    "grid_discards": lambda: cf.parker_modulation_cartesian(small_grid(), kap_rat=0.5, t_limit_years=20.0 / 365.0),
    "guiding_grid": lambda: cf.gc_cartesian(wide_grid(), t_limit_days=0.03),
}


SETUPS.update({"feature_" + n: f for n, f in zip(fs.NAMES, fs.ALL)})
FULL = 66048   # a block of slots beyond one wave per SIMD, from where every kernel's drain is packed


@pytest.mark.parametrize("precision", [E.PREC_FP64, E.PREC_MIXED])
@pytest.mark.parametrize("name", sorted(SETUPS))
def test_records_do_not_depend_on_the_form(name, precision):
    s = SETUPS[name]()
    opt = dict(precision=precision, max_attempts=3)
    full = FULL if name.startswith("feature_") or name in ("guiding", "radial") else MANY
    st, ref = E.Simulation.from_setup(s, graph_launches=1, **opt).run(full, seed=4)
    assert st.done == full
    # the packed drain, the largest run of four lanes, partial waves, resumed streams, one
    for n, spl in ((full, 100), (16384, 2000), (257, 7), (63, 50), (1, 2000)):
        sim = E.Simulation.from_setup(s, steps_per_launch=spl, **opt)
        st, rec = sim.run(n, seed=4)
        assert st.done == n
        for k in E.RECORD_DTYPE.names:
            np.testing.assert_array_equal(rec[k], ref[k][:n], err_msg=f"{name} n={n} {k}")
    print(f"[forms] {name} precision {precision}: {int(ref['steps'].sum())} steps, {int((ref['status'] != 0).sum())} abandoned", flush=True)
