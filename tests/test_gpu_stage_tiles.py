"""Narrow tiles of the LDS super-stages (GPU): the 100-, 125-, 729- and 1000-point
instances on both sides of the rule's line (256 workgroups of the wide tile),
with remainders, and their chirp-source form.  Oracle and bounds as elsewhere.
"""
import numpy as np
import pytest

from flagfft_amd import flagfft as ff

from .helpers import check_accuracy, complex_input, dev_tensor, host, stream_of, sync

pytestmark = pytest.mark.gpu


def _run(gpu, shape, batch, dbl, word):
    t = ff.Type.Z2Z if dbl else ff.Type.C2C
    n = int(np.prod(shape))
    x = complex_input(n + batch, (batch, *shape), np.complex128 if dbl else np.complex64)
    xd = dev_tensor(x, gpu)
    yd, zd = dev_tensor(np.full_like(x, 7.0), gpu), dev_tensor(np.full_like(x, 7.0), gpu)
    with ff.Plan.many(len(shape), list(shape), None, 1, n, None, 1, n, t, batch) as p:
        p.set_stream(stream_of(gpu))
        assert word in p.description(), p.description()
        go = p.z2z if dbl else p.c2c
        go(xd.data_ptr(), yd.data_ptr(), ff.FORWARD)
        go(xd.data_ptr(), zd.data_ptr(), ff.INVERSE)
        sync(gpu)
    ax = tuple(range(1, len(shape) + 1))
    x64 = x.astype(np.complex128)
    check_accuracy(host(yd), np.fft.fftn(x64, axes=ax), t, n, row_len=n, what=f"fwd {shape}")
    check_accuracy(host(zd), np.fft.ifftn(x64, axes=ax) * n, t, n, row_len=n, what=f"inv {shape}")


# rows x columns: the columns run k_stage; 256 C wide-tile units are 8192 (100, 125),
# 4096 (1000) and 2048 (729) in FP32
COLUMNS = [(100, 7), (100, 8191), (100, 8200), (125, 3), (125, 129), (125, 8193), (729, 5), (729, 2047), (729, 2052),
           (1000, 2), (1000, 77), (1000, 4095), (1000, 4100)]


@pytest.mark.parametrize("dbl", [False, True], ids=["fp32", "fp64"])
@pytest.mark.parametrize("rows,cols", COLUMNS)
def test_columns(gpu, rows, cols, dbl):
    rad = {100: "[10x10]", 125: "[5x5x5]", 729: "[9x9x9]", 1000: "[10x10x10]"}[rows]
    _run(gpu, (rows, cols), 1, dbl, rad)


@pytest.mark.parametrize("dbl", [False, True], ids=["fp32", "fp64"])
@pytest.mark.parametrize("n,batch", [(1000000, 1), (1000000, 3), (1000000, 5), (100000, 3), (125000, 1), (531441, 2), (531441, 4)])
def test_chains(gpu, n, batch, dbl):
    _run(gpu, (n,), batch, dbl, "k_stage")


@pytest.mark.parametrize("n,batch", [(1000003, 1)])
def test_chirp_source(gpu, n, batch):
    x = complex_input(n, (batch, n), np.complex64)
    xd = dev_tensor(x, gpu)
    yd = dev_tensor(np.full_like(x, 7.0), gpu)
    with ff.Plan.one_d(n, ff.Type.C2C, batch) as p:
        p.set_stream(stream_of(gpu))
        p.c2c(xd.data_ptr(), yd.data_ptr(), ff.FORWARD)
        sync(gpu)
    check_accuracy(host(yd), np.fft.fft(x.astype(np.complex128), axis=1), ff.Type.C2C, n, row_len=n, what="prime")
