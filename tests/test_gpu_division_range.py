"""The FP64 stage kernel on states whose quotients leave the range its
unchecked divisions are exact in (vh::DivTry: quotients below 2^-950, divisors
outside [2^-16, 2^100]), so that lanes take the checked evaluation: bit for bit
the oracle, for a single event and for the same event in a batch, with such
cells beside ordinary ones in a wave."""
import numpy as np
import pytest

import vhtest as V
from cpuvh_amd import Batch, Hydro

pytestmark = pytest.mark.gpu

FIELDS = ["e", "p", "ut", "ux", "uy", "un", "ttt", "ttx", "tty", "ttn", "pitt", "pitx", "pity", "pitn", "pixx", "pixy",
          "pixn", "piyy", "piyn", "pinn"]


def _ic(kind, shape, lattice, bulk):
    nx, ny, nz = shape
    ic = V.random_ic(nx, ny, nz, 0.1, 0.6, seed=11, lattice=lattice, bulk=bulk)
    rng = np.random.default_rng(5)
    n = nx * ny * nz
    some = rng.random(n) < 0.5
    if kind == "tiny_shear":
        f = np.where(some, 10.0 ** -rng.uniform(280, 305, n), 1.0)
        ic["pi"] = (ic["pi"].reshape(10, n) * f).ravel()
    elif kind == "tiny_flow":
        for c in ("ux", "uy"):
            ic[c] = np.where(some, rng.standard_normal(n) * 10.0 ** -rng.uniform(285, 300, n), ic[c])
        ic["ut"] = np.sqrt(1 + ic["ux"] ** 2 + ic["uy"] ** 2 + 0.36 * ic["un"] ** 2)
    elif kind == "slow_u":  # u^tau outside the divisors' range in a few cells
        ic["ut"] = np.where(rng.random(n) < 0.1, 1e-6, ic["ut"])
    return ic


@pytest.mark.parametrize("kind", ["tiny_shear", "tiny_flow", "slow_u"])
@pytest.mark.parametrize("shape", [(21, 17, 1), (11, 9, 7)])
@pytest.mark.parametrize("lattice,bulk", [(True, True), (False, False)])
def test_bitwise_outside_the_division_range(kind, shape, lattice, bulk):
    print(f"case {kind} {shape} lattice={lattice} bulk={bulk}", flush=True)
    t0, dt, dx = 0.6, 0.02, 0.1
    # a second step from the slow cells reaches e above 2^31 table spacings, where the host's
    # conversion of the table index overflows
    steps = 1 if kind == "slow_u" else 2
    table = V.eos_table() if lattice else None
    ic = _ic(kind, shape, lattice, bulk)
    o = V.Oracle(*shape, dx, dx, dx, dt, t0, 0.2, bulk=bulk, table=table)
    o.set_ic(ic)
    o.init_conserved(t0)
    g = Hydro(*shape, dx, dx, dx, dt, t0, 0.2, bulk=bulk, eos_table=table)
    g.upload_ic(ic["e"], ic["p"], ic["ut"], ic["ux"], ic["uy"], ic["un"], ic["pi"], ic.get("Pi"))
    g.init_conserved(t0)
    b = Batch(shape[0] * shape[1] * shape[2], 1, steps + 1, bulk=bulk, eos_table=table)
    k = b.add(*shape, dx, dx, dx, dt, ic=ic, t0=t0, etabar=0.2)
    for n in range(steps):
        assert o.step(t0 + n * dt) == 0
    g.steps(1, steps)
    b.steps(steps)
    for f in FIELDS + (["Pi"] if bulk else []):
        want = o.get(f)
        assert V.bits_equal(want, g.get(f)), f
        assert V.bits_equal(want, b.get(k, f)), f
    g.close()
