"""How many launches a run that is waited for takes: none to speak of after its trajectories have ended, and whole ones
where no launch could pack its slots.  The records are those of the replayed graph, whatever the rounds."""
import numpy as np
import pytest

import feature_setups as fs
from spectrum_amd import engine as E

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 500, 60000])
@pytest.mark.parametrize("precision", [E.PREC_FP64, E.PREC_MIXED])
def test_run_that_ends_in_its_first_launch(precision, n):
    st, rec = E.Simulation.from_setup(fs.fieldline_spiral(), precision=precision).run(n, seed=2)
    assert int(rec["steps"].max()) <= 2000
    assert st.launches <= 5   # the first, and a round of at most four that bins the events


def test_whole_launches_where_nothing_packs():
    spl = 6000   # the last of three whole launches is two thirds full
    s = fs.gc_qlt_spiral()
    st, rec = E.Simulation.from_setup(s, precision=E.PREC_MIXED, steps_per_launch=spl).run(500, seed=3)
    whole = -(-int(rec["steps"].max()) // spl)
    print(f"[rounds] longest {int(rec['steps'].max())} steps, {st.launches} launches of {spl}", flush=True)
    assert whole >= 2 and st.launches <= whole + 1
    _, ref = E.Simulation.from_setup(s, precision=E.PREC_MIXED, graph_launches=1).run(500, seed=3)
    for k in E.RECORD_DTYPE.names:
        np.testing.assert_array_equal(rec[k], ref[k], err_msg=k)
