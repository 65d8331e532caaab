"""Served queries of one pool that drain together: more slots than the four-lane form takes, so the running slots of
several queries are packed into full waves, with sizes that leave odd parts, different lengths, and a query that
arrives during the drain.  Every result equals the single run's."""
import time

import numpy as np
import pytest

from spectrum_amd import configs as cf
from spectrum_amd import engine as E
from spectrum_amd.server import Server

pytestmark = pytest.mark.gpu


def modulation(days):
    return cf.parker_modulation(n_energies=7, r_start_au=20.0, t_limit_years=days / 365.0, time_action=0)


def shock(days):
    return cf.dsa_shock(t_limit_days=days, src_ratio=1.01)


# the mixed shock has no four-lane form: packed from one wave per SIMD (65536 slots)
CASES = {
    "modulation": (modulation, ((9001, 8.0), (8003, 3.0), (7, 20.0), (20011, 5.0)), (3001, 2.0)),
    "shock": (shock, ((40009, 0.02), (30011, 0.01), (65, 0.05), (7, 0.03)), (1001, 0.01)),
}


@pytest.mark.parametrize("prec", [E.PREC_FP64, E.PREC_MIXED])
@pytest.mark.parametrize("name", sorted(CASES))
def test_mix_that_drains_packed(name, prec):
    make, sizes, late = CASES[name]
    ref, longest = [], 0
    for i, (n, length) in enumerate(sizes + (late,)):
        sim = E.Simulation.from_setup(make(length), precision=prec)
        st, rec = sim.run(n, seed=20 + i)
        assert st.done == n
        longest = max(longest, int(rec["steps"].max()))
        ref.append(sim.distro(0))
    spl = max(1, longest // 60)
    with Server(precision=prec, steps_per_launch=spl) as srv:
        ids = [srv.submit(make(length), n, seed=20 + i) for i, (n, length) in enumerate(sizes)]
        done = lambda: sum(srv.info(q)["done"] for q in ids)
        total = sum(n for n, _ in sizes)
        while done() < total // 2:   # the drain has begun
            time.sleep(1.0e-4)
        ids.append(srv.submit(make(late[1]), late[0], seed=20 + len(sizes)))
        at = done()
        for q in ids:
            assert srv.wait(q, timeout=100.0)
        st = srv.stats()
        assert st["pools"] == 1
        print(f"[packed] {name} precision {prec}: {total} trajectories, {spl} steps a launch of at most {longest}, "
              f"late query at {at} done", flush=True)
        for q, want in zip(ids, ref):
            got = srv.result(q)
            for a, b in zip(got, want):
                np.testing.assert_array_equal(a, b)
