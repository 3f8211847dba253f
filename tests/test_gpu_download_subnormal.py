"""Downloads of a mixed-precision event whose FP32 fields hold subnormal values,
by a thread that takes subnormals as zero in its own arithmetic: the values the
device holds, the same into pageable memory (widened on the host) and into
pinned memory (widened on the device)."""
import numpy as np
import pytest
import torch

import cpuvh_amd as C
import vhtest as V

pytestmark = pytest.mark.gpu


def test_subnormal_fields_cross_whatever_the_threads_mode():
    nx, ny = 33, 21
    n, rng = nx * ny, np.random.default_rng(4)
    e = rng.random(n) + 0.5
    pi = rng.standard_normal((10, n)) * 1e-40
    b = C.Batch(n, 1, 2, precision=C.PREC_MIXED)
    k = b.add(nx, ny, 1, 0.1, 0.1, 0.1, 0.02, ic={"e": e, "p": e / 3, "pi": pi.ravel()}, t0=0.6, etabar=0.2)
    want = {f: b.get(k, f) for f in ("e", "ttt", "pixx", "pixy")}
    assert np.all(np.abs(want["pixx"] - pi[4]) <= 2.0 ** -149) and np.any(want["pixx"] != 0)
    if not torch.set_flush_denormal(True):
        pytest.skip("no flush-to-zero mode")
    try:
        got = {f: b.get(k, f) for f in want}
        t = torch.empty(n, dtype=torch.float64).pin_memory()
        C.Hydro._check(C._lib().vh_batch_download(b.b, k, C.FIELD["pixx"], t.data_ptr()), "download")
        still = float(np.float64(5e-324) * np.float64(1.0))  # the thread's mode is its own again
    finally:
        torch.set_flush_denormal(False)
    for f in want:
        assert V.bits_equal(want[f], got[f]), f
    assert V.bits_equal(want["pixx"], t.numpy())
    assert still == 0.0
    b.close()
