"""Single events at proper times and time steps so small that t, t^2, t^3 or dt
fall far below 1, as divisors of the source terms: bit for bit the oracle."""
import pytest

import vhtest as V
from cpuvh_amd import Hydro

pytestmark = pytest.mark.gpu

FIELDS = ["e", "p", "ut", "ux", "uy", "un", "ttt", "ttx", "tty", "ttn", "pitt", "pitx", "pity", "pitn", "pixx", "pixy",
          "pixn", "piyy", "piyn", "pinn"]


@pytest.mark.parametrize("t0,dt", [(0.02, 5e-4), (1e-3, 1e-5), (1e-5, 1e-9)])
@pytest.mark.parametrize("shape", [(21, 17, 1), (11, 9, 7)])
@pytest.mark.parametrize("lattice", [True, False])
def test_bitwise_at_early_times(t0, dt, shape, lattice):
    print(f"case t0={t0} dt={dt} {shape} lattice={lattice}", flush=True)
    dx, steps = 0.1, 3
    table = V.eos_table() if lattice else None
    ic = V.random_ic(*shape, dx, t0, seed=3, lattice=lattice, pi_scale=1e-4)
    o = V.Oracle(*shape, dx, dx, dx, dt, t0, 0.2, table=table)
    o.set_ic(ic)
    o.init_conserved(t0)
    g = Hydro(*shape, dx, dx, dx, dt, t0, 0.2, eos_table=table)
    g.upload_ic(ic["e"], ic["p"], ic["ut"], ic["ux"], ic["uy"], ic["un"], ic["pi"])
    g.init_conserved(t0)
    for n in range(steps):
        t = t0 + n * dt
        assert o.step(t) == 0
        g.step(t)
        for f in FIELDS:
            assert V.bits_equal(o.get(f), g.get(f)), (f, n)
    g.close()
