"""Two-pass Bluestein convolutions in register-resident launches (GPU).

M = R0 R1: every square convolution instance (R1 = 64, 256, 1024, 4096) with
narrow and wide outer passes, lengths just below M / 2 (the last outputs
before the pruned half), and sequences that share a tile.
Real odd lengths read real / half-spectrum sequences and write the other.
Oracle and bounds as the other length tests.
"""
import numpy as np
import pytest

from flagfft_amd import flagfft as ff
from oracle import oracle as ora

from .helpers import check_accuracy, complex_input, dev_tensor, host, real_input, stream_of, sync

pytestmark = pytest.mark.gpu

# (n, [R0, R1], batch); an explicit split takes effect when M is the first
# 13-smooth length from 2 n - 1 on
CASES = [(32761, [1024, 64], 1), (32761, [256, 256], 5), (32761, [64, 1024], 3), (16381, [128, 256], 2),
         (16381, [32, 1024], 3), (131071, [256, 1024], 2), (65521, [512, 256], 9), (65521, [32, 4096], 1),
         (262139, [512, 1024], 3)]
CASES64 = [(8191, [256, 64], 3), (32761, [256, 256], 2), (16381, [128, 256], 2), (32761, [64, 1024], 3),
           (131071, [256, 1024], 2)]


def _plan(n, passes, t, batch):
    assert ff.set_tuning(passes=passes) == ff.Result.SUCCESS
    try:
        p = ff.Plan.one_d(n, t, batch)
    finally:
        ff.set_tuning()
    desc = p.description()
    assert f"super_radices=[{passes[0]},{passes[1]}]" in desc and "k_col_conv<" in desc and "kernels=3" in desc, desc
    return p


@pytest.mark.parametrize("n,passes,batch,dbl", [c + (False,) for c in CASES] + [c + (True,) for c in CASES64])
def test_complex(gpu, n, passes, batch, dbl):
    t = ff.Type.Z2Z if dbl else ff.Type.C2C
    x = complex_input(n + batch, (batch, n), np.complex128 if dbl else np.complex64)
    xd = dev_tensor(x, gpu)
    for d, sign in ((ff.FORWARD, -1), (ff.INVERSE, 1)):
        yd = xd.clone().zero_()
        with _plan(n, passes, t, batch) as p:
            p.set_stream(stream_of(gpu))
            (p.z2z if dbl else p.c2c)(xd.data_ptr(), yd.data_ptr(), d)
            sync(gpu)
        check_accuracy(host(yd), ora.fft(x.astype(np.complex128), sign), t, n, row_len=n, what=f"{passes} {sign}")


@pytest.mark.parametrize("n,passes,batch,dbl", [(16381, [512, 64], 3, False), (32761, [256, 256], 5, False),
                                                (32761, [64, 1024], 2, False), (262139, [512, 1024], 2, False),
                                                (32761, [256, 256], 2, True), (8191, [256, 64], 7, True)])
def test_real_odd(gpu, n, passes, batch, dbl):
    tf, ti = (ff.Type.D2Z, ff.Type.Z2D) if dbl else (ff.Type.R2C, ff.Type.C2R)
    rdt, cdt = (np.float64, np.complex128) if dbl else (np.float32, np.complex64)
    h = n // 2 + 1
    x = real_input(n, (batch, n), rdt)
    xd = dev_tensor(x, gpu)
    Xd = dev_tensor(np.zeros((batch, h), cdt), gpu)
    with _plan(n, passes, tf, batch) as p:
        p.set_stream(stream_of(gpu))
        (p.d2z if dbl else p.r2c)(xd.data_ptr(), Xd.data_ptr())
        sync(gpu)
    check_accuracy(host(Xd), ora.rfft(x.astype(np.float64)), tf, n, row_len=h, what=f"R2C {passes}")
    # any half spectrum: the oracle's C2R ignores Im of the DC bin
    Y = complex_input(n + 1, (batch, h), cdt)
    Yd = dev_tensor(Y, gpu)
    yd = xd.clone().zero_()
    with _plan(n, passes, ti, batch) as p:
        p.set_stream(stream_of(gpu))
        (p.z2d if dbl else p.c2r)(Yd.data_ptr(), yd.data_ptr())
        sync(gpu)
    assert np.array_equal(host(Yd), Y)
    check_accuracy(host(yd), ora.irfft(Y.astype(np.complex128), n), ti, n, row_len=n, what=f"C2R {passes}")
