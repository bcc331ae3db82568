"""Loads of the register-resident passes (GPU): first and later passes, whole tiles and
the last one that ends partially, in chains of two and three passes, against the
oracle (bounds as elsewhere), with a row past the output that has to stay.
"""
import numpy as np
import pytest

from flagfft_amd import flagfft as ff
from oracle import oracle as ora

from .helpers import check_accuracy, complex_input, dev_tensor, host, stream_of, sync

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("passes,batch,dbl", [([64, 16], 1, False), ([16, 64], 3, False), ([256, 64], 1, False),
                                              ([1024, 16], 1, False), ([32, 128], 2, False), ([512, 256, 16], 1, False),
                                              ([4096, 64], 1, False), ([64, 4096], 1, False), ([2048, 1024], 2, False),
                                              ([256, 25], 1, False), ([64, 81], 5, False), ([256, 64], 3, True),
                                              ([512, 1024], 1, True), ([1024, 64], 2, True), ([128, 81], 3, True)])
def test_passes(gpu, passes, batch, dbl):
    n = int(np.prod(passes))
    t = ff.Type.Z2Z if dbl else ff.Type.C2C
    x = complex_input(n + batch, (batch, n), np.complex128 if dbl else np.complex64)
    xd = dev_tensor(x, gpu)
    yd = dev_tensor(np.full((batch + 1, n), 7.0, x.dtype), gpu)
    assert ff.set_tuning(passes=passes) == ff.Result.SUCCESS
    try:
        p = ff.Plan.one_d(n, t, batch)
    finally:
        ff.set_tuning()
    with p:
        assert "k_col<" in p.description(), p.description()
        p.set_stream(stream_of(gpu))
        (p.z2z if dbl else p.c2c)(xd.data_ptr(), yd.data_ptr(), ff.FORWARD)
        sync(gpu)
    y = host(yd)
    assert np.all(y[batch] == 7.0)
    check_accuracy(y[:batch], ora.fft(x.astype(np.complex128)), t, n, row_len=n, what=f"{passes}")
