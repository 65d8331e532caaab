"""A run of no trajectories: begin, advance and finish succeed and report zeros, with and without a replayed graph, and
the handle runs a following batch as a new one does."""
import numpy as np
import pytest

from spectrum_amd import configs as cf
from spectrum_amd import engine as E

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [E.PREC_FP64, E.PREC_MIXED])
@pytest.mark.parametrize("graph", [0, 2])
@pytest.mark.parametrize("make", [cf.dsa_shock, cf.gc_uniform])
def test_empty_run(make, graph, precision):
    s = make()
    sim = E.Simulation.from_setup(s, precision=precision, graph_launches=graph, steps_per_launch=50)
    for _ in range(2):
        sim.begin(0, seed=1)
        for n in (0, 1, 3):
            st = sim.advance(n)
            assert st.done == 0 and st.steps_executed == 0 and st.failed == 0
        st, _ = sim.finish()
        assert st.done == 0 and st.steps_done == 0
    counts, sums, events = sim.distro(0)
    assert not counts.any() and not sums.any() and events == 0
    st, rec = sim.run(0, seed=1)
    assert st.done == 0 and len(rec) == 0
    sim.begin(300, seed=1)
    sim.advance(4)
    a = sim.distro(0)
    st = E.Simulation.from_setup(s, precision=precision, steps_per_launch=50)
    st.begin(300, seed=1)
    st.advance(4)
    b = st.distro(0)
    np.testing.assert_array_equal(a[0], b[0])
    np.testing.assert_array_equal(a[1], b[1])
