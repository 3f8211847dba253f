"""The FP64 stage kernel where every quotient of the shear terms is subnormal
(shear of 1e-313 to 1e-322, energy and flow ordinary): bit for bit the oracle,
for a single event, and for the same event in a batch."""
import numpy as np
import pytest

import vhtest as V
from cpuvh_amd import Batch, Hydro

pytestmark = pytest.mark.gpu

FIELDS = ["e", "p", "ut", "ux", "uy", "un", "ttt", "ttx", "tty", "ttn", "pitt", "pitx", "pity", "pitn", "pixx", "pixy",
          "pixn", "piyy", "piyn", "pinn"]


@pytest.mark.parametrize("shape", [(41, 37, 1), (21, 17, 9)])
@pytest.mark.parametrize("lattice", [True, False])
@pytest.mark.parametrize("static", [True, False])
def test_bitwise_with_subnormal_shear(shape, lattice, static):
    print(f"case {shape} lattice={lattice} static={static}", flush=True)
    t0, dt, dx, steps = 0.6, 0.02, 0.1, 2
    table = V.eos_table() if lattice else None
    ic = V.random_ic(*shape, dx, t0, seed=11, lattice=lattice)
    n = shape[0] * shape[1] * shape[2]
    r = np.random.default_rng(5)
    if static:  # uniform and at rest: nothing but the shear itself drives the shear
        ic.update(e=np.full(n, 5.0), p=np.full(n, 5.0 / 3.4), ut=np.ones(n), ux=np.zeros(n), uy=np.zeros(n),
                  un=np.zeros(n))
    ic["pi"] = (r.standard_normal((10, n)) * 10.0 ** -r.uniform(313, 322, (10, n))).ravel()
    o = V.Oracle(*shape, dx, dx, dx, dt, t0, 0.2, table=table)
    o.set_ic(ic)
    o.init_conserved(t0)
    g = Hydro(*shape, dx, dx, dx, dt, t0, 0.2, eos_table=table)
    g.upload_ic(ic["e"], ic["p"], ic["ut"], ic["ux"], ic["uy"], ic["un"], ic["pi"])
    g.init_conserved(t0)
    b = Batch(n, 1, steps + 1, eos_table=table)
    k = b.add(*shape, dx, dx, dx, dt, ic=ic, t0=t0, etabar=0.2)
    for s in range(steps):
        assert o.step(t0 + s * dt) == 0
        g.step(t0 + s * dt)
        b.steps(1)
        for f in FIELDS:
            want = o.get(f)
            assert V.bits_equal(want, g.get(f)), (f, s)
            assert V.bits_equal(want, b.get(k, f)), (f, s)
    g.close()
    b.close()
