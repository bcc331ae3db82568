"""LDS Bluestein convolutions over workgroups, by source (GPU): contiguous complex, real
and Hermitian sequences and strided ones, at the ends of a block (n just past M / 4 and
just under M / 2 of the split in 4), with values past the sequence that must not
come in.  Oracle numpy in 64 bits, bounds as elsewhere.
"""
import numpy as np
import pytest

from flagfft_amd import flagfft as ff

from .helpers import check_accuracy, complex_input, dev_tensor, host, real_input, stream_of, sync

pytestmark = pytest.mark.gpu

# M = 16384 (n 4099 .. 8187), 20160 (.. 10079), FP64 8192, 10080
LENGTHS = [(4099, 3, False), (8187, 5, False), (7919, 64, False), (10007, 33, False), (10079, 2, False),
           (15013, 9, False), (2503, 40, True), (4093, 64, True), (5003, 7, True), (10007, 17, True)]


@pytest.mark.parametrize("n,batch,dbl", LENGTHS)
def test_real_and_half_spectrum(gpu, n, batch, dbl):
    tf, ti = (ff.Type.D2Z, ff.Type.Z2D) if dbl else (ff.Type.R2C, ff.Type.C2R)
    rdt, cdt = (np.float64, np.complex128) if dbl else (np.float32, np.complex64)
    h = n // 2 + 1
    x, Y = real_input(n, (batch, n), rdt), complex_input(n + 1, (batch, h), cdt)
    xd, Yd = dev_tensor(x, gpu), dev_tensor(Y, gpu)
    Xd, yd = dev_tensor(np.full((batch, h), 7.0, cdt), gpu), dev_tensor(np.full((batch, n), 7.0, rdt), gpu)
    with ff.Plan.one_d(n, tf, batch) as pf, ff.Plan.one_d(n, ti, batch) as pi:
        for p, src in ((pf, 1), (pi, 2)):
            p.set_stream(stream_of(gpu))
            assert "k_bluestein_split<" in p.description() and f",{src}>[" in p.description(), p.description()
        (pf.d2z if dbl else pf.r2c)(xd.data_ptr(), Xd.data_ptr())
        (pi.z2d if dbl else pi.c2r)(Yd.data_ptr(), yd.data_ptr())
        sync(gpu)
    check_accuracy(host(Xd), np.fft.rfft(x.astype(np.float64), axis=1), tf, n, row_len=h, what="R2C")
    Y64 = Y.astype(np.complex128)
    Y64[:, 0] = Y64[:, 0].real  # Im of the DC bin does not count
    check_accuracy(host(yd), np.fft.irfft(Y64, n, axis=1) * n, ti, n, row_len=n, what="C2R")


@pytest.mark.parametrize("n,batch,stride", [(8187, 3, 1), (8187, 3, 2), (10007, 33, 3)])
def test_strided_with_neighbours(gpu, n, batch, stride):
    """Elements between and past the sequences hold infinities."""
    t = ff.Type.C2C
    x = complex_input(n + stride, (batch, n), np.complex64)
    dist = n * stride + 5
    buf = np.full(batch * dist, np.inf + 1j * np.inf, np.complex64)
    for b in range(batch):
        buf[b * dist:b * dist + n * stride:stride] = x[b]
    xd, yd = dev_tensor(buf, gpu), dev_tensor(np.full((batch, n), 7.0, np.complex64), gpu)
    with ff.Plan.many_ext(1, [n], [n], stride, dist, [n], 1, n, t, batch) as p:
        p.set_stream(stream_of(gpu))
        assert f",{0 if stride == 1 else 3}>[" in p.description(), p.description()
        p.c2c(xd.data_ptr(), yd.data_ptr(), ff.FORWARD)
        sync(gpu)
    check_accuracy(host(yd), np.fft.fft(x.astype(np.complex128), axis=1), t, n, row_len=n, what=f"stride {stride}")
