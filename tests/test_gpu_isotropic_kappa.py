"""kappa isotropic and a function of |x| alone: the step forms div(kappa) without the magnetic field, on the solar
wind and on the grid.  FP64 parity with the oracle, which evaluates the whole stencil, for every branch of the power
(2, 1, 0, 1/2, general), with one lane and with four per trajectory, and where the path must not be taken: a Larmor
radius of the order of the distance to the Sun."""
import os

import numpy as np
import pytest

from spectrum_amd import cartesian
from spectrum_amd import configs as cf
from spectrum_amd import engine as E
from spectrum_amd.data_container import DataContainer
from test_gpu_parity import check_parity, sensitivity

pytestmark = pytest.mark.gpu
THREADS = min(16, os.cpu_count() or 1)


def setup(exponent, grid, B_nT):
    s = cf.parker_modulation_radial(n_energies=4, inner_au=0.3, outer_au=5.0, T1_MeV=100.0, grid=cartesian.parker_spiral(12, 30.0) if grid else None)
    dif = DataContainer().insert_double(1.5e22 / cf.unit_diffusion).insert_double(cf.GeV).insert_double(cf.one_au)
    dif.insert_double(1.0).insert_double(exponent).insert_double(1.0).insert_int(0)
    dif.insert_double(1.0).insert_double(0.0).insert_double(1.0)
    s.plugins = [(r, n, dif.bytes() if r == cf.DIFFUSION else b) for r, n, b in s.plugins]
    if not grid:
        s.plugins = [(r, n, cf.solarwind(B_nT_1au=B_nT).bytes() if r == cf.BACKGROUND else b) for r, n, b in s.plugins]
    return s


@pytest.mark.parametrize("grid,B_nT", [(False, 5.0), (False, 1e-4), (True, 5.0)])
@pytest.mark.parametrize("exponent", [2.0, 1.0, 0.0, 0.5, 1.3])
def test_fp64_parity(oracle_mod, exponent, grid, B_nT):
    s = setup(exponent, grid, B_nT)
    n = 192
    o = oracle_mod.Oracle(s)
    _, orec = o.run(n, seed=8, threads=THREADS)
    _, prec = oracle_mod.Oracle(s, oracle_mod.FMA_LIB_PATH).run(n, seed=8, threads=THREADS)
    recs = []
    for graph in (0, 1):   # four lanes per trajectory; one
        sim = E.Simulation.from_setup(s, precision=E.PREC_FP64, graph_launches=graph)
        st, rec = sim.run(n, seed=8)
        check_parity(st, rec, orec, sim, o, n, sens=sensitivity(orec, prec))
        recs.append(rec)
    for k in E.RECORD_DTYPE.names:
        np.testing.assert_array_equal(recs[0][k], recs[1][k], err_msg=k)
