"""Tiles of the register-resident column passes at their edges (GPU).

A tile of C adjacent columns may run over the end of one slab into the next
ones and past the last column; launches of few columns take narrower tiles.
Shapes: R columns of w elements in n0 slabs, with w below, just past and far
from a multiple of every tile width, for every super-radix.  Oracle and bounds
as the other rank-3 tests (FP32 2e-6 log2 N, FP64 1e-14 log2 N relative L2).
"""
import numpy as np
import pytest

from flagfft_amd import flagfft as ff
from oracle import oracle as ora

from .helpers import check_accuracy, complex_input, dev_tensor, host, stream_of, sync

pytestmark = pytest.mark.gpu

CASES = [(3, r, w, False) for r in (16, 32, 64, 128, 256, 512, 1024) for w in (3, 33)]
CASES += [(9, 64, 129, False), (37, 64, 7, False), (7, 256, 129, False), (300, 64, 65, False), (33, 1024, 70, False),
          (2, 2048, 1030, False), (2, 2048, 20, False), (2, 4096, 1029, False)]
CASES += [(3, r, w, True) for r in (64, 128, 256, 512, 1024) for w in (5, 17)]
CASES += [(9, 512, 129, True), (5, 1024, 250, True)]


@pytest.mark.parametrize("n0,r,w,dbl", CASES)
def test_columns_over_slab_ends(gpu, n0, r, w, dbl):
    n = n0 * r * w
    t = ff.Type.Z2Z if dbl else ff.Type.C2C
    x = complex_input(n + r, (1, n0, r, w), np.complex128 if dbl else np.complex64)
    xd = dev_tensor(x, gpu)
    yd = xd.clone().zero_()
    guard = yd.clone()  # an untouched neighbour of the output
    with ff.Plan.three_d(n0, r, w, t, 1) as p:
        p.set_stream(stream_of(gpu))
        (p.z2z if dbl else p.c2c)(xd.data_ptr(), yd.data_ptr(), ff.FORWARD)
        sync(gpu)
    assert not bool(guard.abs().any())
    check_accuracy(host(yd), ora.fft3(x.astype(np.complex128)), t, n, row_len=n, factor=2.0, what=f"{n0}x{r}x{w}")


@pytest.mark.parametrize("n,batch,dbl", [(3 * 1024, 3, True), (5 * 1024 * 64, 3, False), (2048 * 1024, 1, False),
                                         (2048 * 1024, 3, False), (1 << 20, 1, False), (1 << 18, 3, True),
                                         (1 << 16, 1, False), (1 << 19, 1, True)])
def test_chains_of_narrow_and_straddling_tiles(gpu, n, batch, dbl):
    """1D chains whose units per sequence are no multiple of the tile, or few enough for the narrow tiles."""
    t = ff.Type.Z2Z if dbl else ff.Type.C2C
    x = complex_input(n + batch, (batch, n), np.complex128 if dbl else np.complex64)
    xd = dev_tensor(x, gpu)
    yd = xd.clone().zero_()
    with ff.Plan.one_d(n, t, batch) as p:
        p.set_stream(stream_of(gpu))
        (p.z2z if dbl else p.c2c)(xd.data_ptr(), yd.data_ptr(), ff.FORWARD)
        sync(gpu)
    check_accuracy(host(yd), ora.fft(x.astype(np.complex128)), t, n, row_len=n, what=f"n={n} batch={batch}")
