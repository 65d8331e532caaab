"""A served query that ends in SetStart (every start lies outside its grid) is complete, and its memory returned, in the
launch that starts it, while another query of the same pool runs on: its waves must have left it by then."""
import numpy as np
import pytest

from spectrum_amd import cartesian
from spectrum_amd import configs as cf
from spectrum_amd import engine as E
from spectrum_amd.server import Server

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [E.PREC_FP64, E.PREC_MIXED])
def test_query_of_failing_starts(prec):
    long_q = cf.gc_cartesian(cartesian.parker_spiral(12, 100.0), t_limit_days=1.0)
    failing = cf.gc_cartesian(cartesian.parker_spiral(6, 6.0), t_limit_days=1.0, r_start_au=50.0)
    n = 3001
    sim = E.Simulation.from_setup(long_q, precision=prec)
    st, _ = sim.run(n, seed=5, records=False)
    assert st.done == n and st.failed == 0
    with Server(precision=prec, steps_per_launch=50) as srv:
        a = srv.submit(long_q, n, seed=5)
        bad = [srv.submit(failing, m, seed=6) for m in (1, 64, 300, 5000)]
        for q, m in zip(bad, (1, 64, 300, 5000)):
            assert srv.wait(q, timeout=60.0)
            info = srv.info(q)
            assert info["failed"] == m and info["steps_executed"] == 0
            srv.release(q)
        assert srv.info(a)["state"] == "running"
        assert srv.wait(a, timeout=100.0)
        for got, want in zip(srv.result(a), sim.distro(0)):
            np.testing.assert_array_equal(got, want)
