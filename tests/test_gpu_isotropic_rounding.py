"""The isotropic kappa(|x|) path, the general stencil and the forms of the step kernel give the same records, bit for bit.

The general stencil runs the same kappa through the stream-dependent branch of the reference's class
(src/diffusion_other.cc:713-723): below its r0 that branch is kap0 (T / T0)^a (r / r0)^b too, and an r0 larger by
2^6 with kap0 larger by 2^(6 b) scales every factor by a power of two, so kappa is the same number.  A last-bit
difference of |x|^2 reaches the FP32 radius about once in 10^9 evaluations: the mixed runs are long enough to meet some."""
import numpy as np
import pytest

from spectrum_amd import cartesian
from spectrum_amd import configs as cf
from spectrum_amd import engine as E
from spectrum_amd.data_container import DataContainer

pytestmark = pytest.mark.gpu
SHIFT = 6


def setup(exponent, grid=None, general=False, inner=0.3, outer=5.0, sw=None):
    s = cf.parker_modulation_radial(n_energies=4, inner_au=inner, outer_au=outer, T1_MeV=100.0, grid=grid)
    k = SHIFT if general else 0
    dif = DataContainer().insert_double(1.5e22 / cf.unit_diffusion * 2.0 ** (k * exponent)).insert_double(cf.GeV).insert_double(cf.one_au * 2.0 ** k)
    dif.insert_double(1.0).insert_double(exponent).insert_double(1.0).insert_int(1 if general else 0)
    dif.insert_double(1.0).insert_double(0.0).insert_double(1.0)
    new = {cf.DIFFUSION: dif.bytes()}
    if sw is not None:
        new[cf.BACKGROUND] = sw.bytes()
    s.plugins = [(r, n, new.get(r, b)) for r, n, b in s.plugins]
    return s


def same(a, b, what):
    for k in E.RECORD_DTYPE.names:
        np.testing.assert_array_equal(a[k], b[k], err_msg=f"{what} {k}")


def run(s, n, precision, first=0, seed=8, **opt):
    st, rec = E.Simulation.from_setup(s, precision=precision, **opt).run(n, seed=seed, first=first)
    assert st.done == n
    return st, rec


@pytest.mark.parametrize("precision", [E.PREC_FP64, E.PREC_MIXED])
@pytest.mark.parametrize("gridded", [False, True])
@pytest.mark.parametrize("exponent", [2.0, 1.0, 0.0, 0.5])
def test_isotropic_path_is_the_general_stencil(exponent, gridded, precision):
    grid = cartesian.parker_spiral(12, 30.0) if gridded else None
    n = 4097
    _, ref = run(setup(exponent, grid, general=True), n, precision, graph_launches=1)
    for graph in (1, 0):   # one lane per trajectory, four
        _, rec = run(setup(exponent, grid), n, precision, graph_launches=graph)
        same(rec, ref, f"graph {graph}")


@pytest.mark.parametrize("precision", [E.PREC_FP64, E.PREC_MIXED])
@pytest.mark.parametrize("exponent", [2.0, 0.5])
def test_guard_on_the_stencil_length(exponent, precision):
    """The isotropic path is refused where the stencil's half length h exceeds |x| / 2.  In a field this weak the Larmor
    radius is several au and more, so h = min(0.6 |x|, 1 au): refused below 2 au, taken above."""
    sw = cf.solarwind(B_nT_1au=1.0e-4, dmax0=cf.one_au, dmax_fraction=0.6)
    n = 4097
    st, ref = run(setup(exponent, general=True, sw=sw), n, precision, graph_launches=1)
    r0 = np.linalg.norm(ref["pos0"], axis=1) / cf.one_au
    r1 = np.linalg.norm(ref["pos"], axis=1) / cf.one_au
    p = ref["mom0"][:, 0].min()
    larmor = p * cf.c_code / (1.0e-13 * 1.0e4 / cf.unit_magnetic) / cf.one_au   # at 1 au; it grows with the distance squared
    assert larmor * 0.3 ** 2 > 1.0 and (r0 < 2.0).all() and (r1 > 4.0).sum() > 100   # these cross 2 au
    for graph in (1, 0):
        _, rec = run(setup(exponent, sw=sw), n, precision, graph_launches=graph)
        same(rec, ref, f"graph {graph}")


@pytest.mark.parametrize("gridded", [False, True])
def test_mixed_long(gridded):
    """Several 10^9 steps: the general stencil and the isotropic path with one lane, and with four in runs that fit
    that form for the first part of them."""
    grid = cartesian.parker_spiral(25, 100.0) if gridded else None
    few, n = 16384, 16 * 16384
    iso, general = (E.Simulation.from_setup(setup(2.0, grid, general=g, inner=0.05, outer=60.0), precision=E.PREC_MIXED, graph_launches=1)
                    for g in (False, True))
    quad = E.Simulation.from_setup(setup(2.0, grid, inner=0.05, outer=60.0), precision=E.PREC_MIXED)
    steps = 0
    for part in range(24):
        st, ref = general.run(n, seed=8, first=part * n)
        steps += int(st.steps_done)
        _, rec = iso.run(n, seed=8, first=part * n)
        same(rec, ref, f"one lane, part {part}")
        for first in range(0, n if part < 2 else 0, few):
            _, rec = quad.run(few, seed=8, first=part * n + first)
            same(rec, ref[first:first + few], f"four lanes, part {part} from {first}")
    print(f"[isotropic] {steps} steps", flush=True)
