"""Mixed 3+1D events of few cells a row, on the tile the batch picks by itself:
the bits of every tile variant set by hand, alone and beside a wider event."""
import numpy as np
import pytest

import vhtest as V
from cpuvh_amd import Batch, PREC_MIXED

pytestmark = pytest.mark.gpu
FIELDS = ["e", "ut", "ux", "un", "ttt", "pixy", "pinn"]


def _run(shapes, lattice, tiles):
    b = Batch(sum(x * y * z for x, y, z in shapes), len(shapes), 8, bulk=True,
              eos_table=V.eos_table() if lattice else None, precision=PREC_MIXED)
    if tiles is not None:
        b.set_tiles(*tiles)
    ids = []
    for k, (nx, ny, nz) in enumerate(shapes):
        ic = V.random_ic(nx, ny, nz, 0.1, 0.6, seed=3 + k, lattice=lattice, bulk=True, flow=0.05, pi_scale=1e-3)
        ids.append(b.add(nx, ny, nz, 0.1, 0.1, 0.1, 0.02, 0.6, 0.1, ic))
    b.steps(4)
    out = [b.get(i, f) for i in ids for f in FIELDS]
    b.close()
    return out


@pytest.mark.parametrize("shapes", [[(5, 9, 7)], [(6, 7, 13)], [(17, 9, 7)], [(20, 5, 5)], [(8, 8, 4)], [(101, 5, 6)],
                                    [(3, 3, 2)], [(17, 13, 9), (40, 11, 5)]])
@pytest.mark.parametrize("lattice", [True, False])
def test_own_choice_has_every_variants_bits(shapes, lattice):
    print(f"case {shapes} lattice={lattice}", flush=True)
    own = _run(shapes, lattice, None)
    assert all(np.isfinite(x).all() for x in own)
    for v in range(3):
        for a, c in zip(own, _run(shapes, lattice, (0, v))):
            assert V.bits_equal(a, c), v
