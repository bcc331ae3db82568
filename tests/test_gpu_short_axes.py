"""Axes of 1 to 9 elements, whose tiles hold one to a few elements per thread of the
run-time-radix pass, with a partial last tile (GPU, float64 oracle).
"""
import numpy as np
import pytest

from flagfft_amd import flagfft as ff

from .helpers import check_accuracy, complex_input, dev_tensor, host, stream_of, sync

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n0", [1, 2, 3, 4, 5, 6, 7, 8, 9])
@pytest.mark.parametrize("n1,n2", [(37, 100), (1, 1), (64, 64)])
@pytest.mark.parametrize("t", ["C2C", "Z2Z"])
def test_short_outer_axis(gpu, n0, n1, n2, t):
    ty = ff.Type[t]
    dt = np.complex64 if t == "C2C" else np.complex128
    x = complex_input(n0 + n1, (n0, n1, n2), dt)
    xd = dev_tensor(x, gpu)
    # (room past the result, which has to stay as it is)
    yd = dev_tensor(np.full(x.size + 8192, 7.0, dt), gpu)
    with ff.Plan.three_d(n0, n1, n2, ty) as p:
        p.set_stream(stream_of(gpu))
        for sign in (ff.FORWARD, ff.INVERSE):
            (p.c2c if t == "C2C" else p.z2z)(xd.data_ptr(), yd.data_ptr(), sign)
            sync(gpu)
            y, x64 = host(yd), x.astype(np.complex128)
            assert (y[x.size:] == 7.0).all()
            ref = np.fft.fftn(x64) if sign == ff.FORWARD else np.fft.ifftn(x64) * x.size
            check_accuracy(y[:x.size].reshape(x.shape), ref, ty, x.size, row_len=x.size)
