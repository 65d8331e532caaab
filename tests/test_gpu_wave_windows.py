"""A run with more waves than the device holds covers whole sets of resident waves per launch, the windows following
each other around the slots: the same records, bit for bit, as launches over every slot (what a replayed graph runs),
from one wave more than a set to a last set that is nearly full, the last wave partly empty."""
import numpy as np
import pytest

from spectrum_amd import cartesian
from spectrum_amd import configs as cf
from spectrum_amd import engine as E

pytestmark = pytest.mark.gpu

SETUPS = {
    "guiding": lambda: cf.gc_diff_scatt(t_limit_days=0.03),
    "modulation": lambda: cf.parker_modulation(n_energies=7, r_start_au=20.0, t_limit_years=8.0 / 365.0, time_action=0),
    "shock_source": lambda: cf.dsa_shock(t_limit_days=0.005, src_ratio=1.01),
    "grid": lambda: cf.parker_modulation_cartesian(cartesian.parker_spiral(12, 100.0), t_limit_years=2.0 / 365.0),
}


@pytest.mark.parametrize("precision", [E.PREC_FP64, E.PREC_MIXED])
@pytest.mark.parametrize("name", sorted(SETUPS))
def test_records_do_not_depend_on_the_windows(name, precision):
    s = SETUPS[name]()
    # sets of 1 to 8 waves per SIMD on 1024 SIMDs are multiples of 65536 slots
    sizes = (131072 + 1, 262144 + 65, 262144 + 48000)
    st, ref = E.Simulation.from_setup(s, precision=precision, graph_launches=1).run(max(sizes), seed=5)
    assert st.done == max(sizes)
    for n in sizes:
        st, rec = E.Simulation.from_setup(s, precision=precision, steps_per_launch=20).run(n, seed=5)
        assert st.done == n
        for k in E.RECORD_DTYPE.names:
            np.testing.assert_array_equal(rec[k], ref[k][:n], err_msg=f"{name} n={n} {k}")
    print(f"[windows] {name} precision {precision}: {int(ref['steps'].sum())} steps", flush=True)
