"""Surface calls with less room than the surface needs (vh_fo_surface,
vh_batch_fo_surface): VH_ERR_CAPACITY with the total and every cube's count, the
arrays left alone, and the wrappers' second call gives what a call with room
gives."""
import ctypes

import numpy as np
import pytest

import cpuvh_amd as C
import vhtest as V

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(25, 23, 1), (15, 13, 9)])
def test_a_second_call_where_the_room_was_too_small(shape):
    print(f"case {shape}", flush=True)
    table = V.eos_table()
    ic = V.random_ic(*shape, 0.1, 0.6, seed=9, lattice=True, bulk=True, e_scale=6.0, e_floor=0.3)
    h = C.Hydro(*shape, 0.1, 0.1, 0.1, 0.02, 0.6, 0.1, T_reg_GeV=0.1, bulk=True, eos_table=table)
    h.upload_ic(ic["e"], ic["p"], ic["ut"], ic["ux"], ic["uy"], ic["un"], ic["pi"], ic["Pi"])
    h.init_conserved(0.6)
    b = C.Batch(h.N, 1, 8, bulk=True, eos_table=table, fo_vars=True)
    k = b.add(*shape, 0.1, 0.1, 0.1, 0.02, 0.6, 0.1, ic, T_reg_GeV=0.1)
    dim = 4 if shape[2] > 1 else 3
    w = np.array([0.04, 0.1, 0.1, 0.1])[:dim]
    eF = h.eos_energy_density(0.15 / V.HBARC)
    n = len(h.fo_flag_ids(eF))
    assert n == len(b.fo_flag_ids(k, eF))
    counts = np.zeros(n, dtype=np.int32)
    p = lambda a: a.ctypes.data  # noqa: E731
    for call, whole in [(lambda *o: C._lib().vh_fo_surface(h.h, p(w), p(counts), *o), h.fo_surface(w)),
                        (lambda *o: C._lib().vh_batch_fo_surface(b.b, k, p(w), p(counts), *o), b.fo_surface(k, w))]:
        total = len(whole[1])
        assert total > 20
        el, var, got = np.full((total, 2 * dim), -7.0), np.full((total, 10), -7.0), ctypes.c_int64()
        counts[:] = -1
        assert call(p(el), p(var), total - 1, ctypes.byref(got)) == C.VH_ERR_CAPACITY
        assert got.value == total and np.array_equal(counts, whole[0]) and np.all(el == -7.0) and np.all(var == -7.0)
        # room for two elements, then for all of them
        m, el, var = C._fo_surface(call, "surface", -7, dim)
        assert m == total and np.array_equal(counts, whole[0])
        assert V.bits_equal(el[:m], whole[1]) and V.bits_equal(var[:m], whole[2])
    h.close()
    b.close()
