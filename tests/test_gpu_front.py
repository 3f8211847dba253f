"""A hot region in a uniform medium: ahead of it velocity and shear fall to the
smallest numbers within a few tens of cells, and the stage kernel's quotients with
them.  Bit for bit the oracle after every few steps."""
import numpy as np
import pytest

import vhtest as V
from cpuvh_amd import Hydro

pytestmark = pytest.mark.gpu

FIELDS = ["e", "ut", "ux", "uy", "un", "ttt", "ttx", "tty", "ttn", "pitt", "pitx", "pity", "pitn", "pixx", "pixy", "pixn",
          "piyy", "piyn", "pinn"]


@pytest.mark.parametrize("shape,steps", [((81, 69, 1), 24), ((41, 37, 33), 8)])
@pytest.mark.parametrize("lattice,bulk", [(True, True), (False, False)])
def test_bitwise_through_the_front(shape, steps, lattice, bulk):
    print(f"case {shape} lattice={lattice} bulk={bulk}", flush=True)
    t0, dt, dx = 0.6, 0.02, 0.1
    table = V.eos_table() if lattice else None
    x, y, z = ((np.arange(n) - (n - 1) / 2) * dx for n in shape)
    Z, Y, X = np.meshgrid(z, y, x, indexing="ij")
    r2 = np.minimum((X ** 2 + Y ** 2 + Z ** 2) / 0.5 ** 2, 1.0)
    e = (0.5 + 5.0 * (1.0 - r2) ** 2).ravel()
    one, nil = np.ones_like(e), np.zeros_like(e)
    ic = {"e": e, "p": e / 3.3, "ut": one, "ux": nil, "uy": nil, "un": nil, "pi": np.zeros(10 * e.size)}
    o = V.Oracle(*shape, dx, dx, dx, dt, t0, 0.1, bulk=bulk, table=table)
    o.set_ic(ic)
    o.init_conserved(t0)
    g = Hydro(*shape, dx, dx, dx, dt, t0, 0.1, bulk=bulk, eos_table=table)
    g.upload_ic(ic["e"], ic["p"], None, None, None, None, None)
    g.init_conserved(t0)
    small = 0
    for n in range(steps):
        assert o.step(t0 + n * dt) == 0
        g.step(t0 + n * dt)
        if n % 4 == 3:
            for f in FIELDS + (["Pi"] if bulk else []):
                want = o.get(f)
                assert V.bits_equal(want, g.get(f)), (f, n)
                small += int(np.sum((want != 0) & (np.abs(want) < 1e-290)))
    assert small > 0
    g.close()
