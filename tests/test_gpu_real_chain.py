"""Even real lengths whose n/2-point chain has the split-spectrum pass in its last
(R2C) or first (C2R) launch (GPU).

Every fused super-radix, wide and narrow tiles, unit 0 and the middle unit (their
own mirror units), the DC, middle and Nyquist bins, padded in-place rows, and
spectra that no real signal has (Im of X_0 and X_h ignored).  Oracle and bounds
as the other real-length tests.
"""
import numpy as np
import pytest

from flagfft_amd import flagfft as ff
from oracle import oracle as ora

from .helpers import check_accuracy, complex_input, dev_tensor, host, real_input, stream_of, sync

pytestmark = pytest.mark.gpu

# (n, batch, super-radices of n / 2 or None); the fused launch is the last of the
# forward chain and the first of the inverse one
FUSED = {False: (64, 128, 256, 512, 1024, 2048), True: (64, 128, 256, 512, 1024)}
CASES = [(1 << 15, 3, [256, 64]), (1 << 15, 2, [64, 256]), (1 << 15, 2, [128, 128]), (1 << 17, 1, None),
         (1 << 17, 40, None), (1 << 18, 2, [256, 512]), (1 << 18, 2, [512, 256]), (1 << 20, 1, None), (1 << 20, 9, None),
         (1 << 21, 1, [1024, 1024]), (1 << 21, 5, [1024, 1024]), (3 << 16, 2, [96, 1024]), (1 << 21, 1, [64, 128, 128]),
         (1 << 22, 4, [1024, 2048]), (1 << 22, 4, [2048, 1024])]


@pytest.mark.parametrize("dbl", [False, True], ids=["fp32", "fp64"])
@pytest.mark.parametrize("n,batch,passes", CASES)
def test_even_real_chain(gpu, n, batch, passes, dbl):
    if dbl and n * batch > 1 << 22:
        batch = 2
    h = n // 2
    tf, ti = (ff.Type.D2Z, ff.Type.Z2D) if dbl else (ff.Type.R2C, ff.Type.C2R)
    rdt, cdt = (np.float64, np.complex128) if dbl else (np.float32, np.complex64)
    x = real_input(n + batch, (batch, n), rdt)
    Y = complex_input(n + 1, (batch, h + 1), cdt)
    xd, Yd = dev_tensor(x, gpu), dev_tensor(Y, gpu)
    Xd = dev_tensor(np.full((batch, h + 1), 7.0, cdt), gpu)
    yd = dev_tensor(np.full((batch, n), 7.0, rdt), gpu)
    if passes:
        assert ff.set_tuning(passes=passes) == ff.Result.SUCCESS
    try:
        with ff.Plan.one_d(n, tf, batch) as pf, ff.Plan.one_d(n, ti, batch) as pi:
            for p, word, end in ((pf, "post", -1), (pi, "pre", 0)):
                p.set_stream(stream_of(gpu))
                if passes is None or passes[end] in FUSED[dbl]:
                    assert f",{word}>" in p.description() and "k_real_" not in p.description(), p.description()
                else:
                    assert f"k_real_{word}" in p.description(), p.description()
            (pf.d2z if dbl else pf.r2c)(xd.data_ptr(), Xd.data_ptr())
            (pi.z2d if dbl else pi.c2r)(Yd.data_ptr(), yd.data_ptr())
            sync(gpu)
    finally:
        ff.set_tuning()
    check_accuracy(host(Xd), ora.rfft(x.astype(np.float64)), tf, n, row_len=h + 1, what=f"R2C {passes}")
    check_accuracy(host(yd), ora.irfft(Y.astype(np.complex128), n), ti, n, row_len=n, what=f"C2R {passes}")
    assert np.array_equal(host(Yd), Y) and np.array_equal(host(xd), x)


@pytest.mark.parametrize("n,batch", [(1 << 17, 3), (1 << 20, 2)])
def test_in_place_padded_rows(gpu, n, batch):
    h = n // 2
    x = real_input(n, (batch, n), np.float32)
    buf = np.zeros((batch, 2 * (h + 1)), np.float32)
    buf[:, :n] = x
    d = dev_tensor(buf, gpu)
    with ff.Plan.many(1, [n], [2 * (h + 1)], 1, 2 * (h + 1), [h + 1], 1, h + 1, ff.Type.R2C, batch) as pf, \
            ff.Plan.many(1, [n], [h + 1], 1, h + 1, [2 * (h + 1)], 1, 2 * (h + 1), ff.Type.C2R, batch) as pi:
        for p in (pf, pi):
            p.set_stream(stream_of(gpu))
            assert "k_col_real<" in p.description()
        pf.r2c(d.data_ptr(), d.data_ptr())
        sync(gpu)
        X = host(d).view(np.complex64).reshape(batch, h + 1)
        check_accuracy(X, ora.rfft(x.astype(np.float64)), ff.Type.R2C, n, row_len=h + 1, what="in place R2C")
        pi.c2r(d.data_ptr(), d.data_ptr())
        sync(gpu)
    check_accuracy(host(d)[:, :n], x.astype(np.float64) * n, ff.Type.C2R, n, row_len=n, factor=2.0, what="in place C2R")
