"""Downloads through the pinned chunks (vh::HostCopy: 131,072 doubles each) at
the chunks' edges, and into memory the runtime knows, which is copied to
directly: the same values either way, in FP64 and widened from the mixed form's
FP32 (with the low parts of T^{tau mu})."""
import numpy as np
import pytest
import torch

import cpuvh_amd as C
import vhtest as V

pytestmark = pytest.mark.gpu


def _pinned(call, owner, n):
    t = torch.empty(n, dtype=torch.float64).pin_memory()
    C.Hydro._check(call(*owner, t.data_ptr()), "download")
    return t.numpy().copy()


@pytest.mark.parametrize("nx,ny", [(3, 3), (512, 256), (513, 256), (512, 513), (1023, 385)])
def test_downloads_at_chunk_edges(nx, ny):
    print(f"case {nx} x {ny}", flush=True)
    n, L = nx * ny, C._lib()
    rng = np.random.default_rng(7)
    e = (rng.random(n) + 0.5).astype(np.float32).astype(np.float64)
    g = C.Hydro(nx, ny, 1, 0.1, 0.1, 0.1, 0.02, 0.6, 0.2)
    g.upload_ic(e, e / 3, None, None, None, None, None)
    assert V.bits_equal(g.get("e"), e) and V.bits_equal(g.get("p"), e / 3)
    assert V.bits_equal(_pinned(L.vh_download, (g.h, C.FIELD["p"]), n), e / 3)
    g.close()
    for precision in (C.PREC_FP64, C.PREC_MIXED):
        b = C.Batch(n + 9, 2, 2, precision=precision)
        b.add(3, 3, 1, 0.1, 0.1, 0.1, 0.02, ic={"e": e[:9], "p": e[:9] / 3}, t0=0.6, etabar=0.2)
        k = b.add(nx, ny, 1, 0.1, 0.1, 0.1, 0.02, ic={"e": e, "p": e / 3}, t0=0.6, etabar=0.2)
        assert V.bits_equal(b.get(k, "e"), e)
        ttt = b.get(k, "ttt")  # (e + p) - p; the mixed form's hi + lo hold it to about 2^-48
        assert np.max(np.abs(ttt - e)) <= 2.0 ** -44
        for f in ("e", "ttt"):
            assert V.bits_equal(_pinned(L.vh_batch_download, (b.b, k, C.FIELD[f]), n), b.get(k, f)), (precision, f)
        b.close()
