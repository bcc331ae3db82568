"""LDS Bluestein convolutions spread over workgroups (GPU): sequence counts that are
no multiple of 8 (whose last blocks map to workgroups another way) and both sides of
the rule's lines (1/8 and 1/4 of 256 CUs).  Oracle numpy in 64 bits, bounds as
elsewhere.
"""
import numpy as np
import pytest

from flagfft_amd import flagfft as ff

from .helpers import check_accuracy, complex_input, dev_tensor, host, stream_of, sync

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,batch,dbl,split", [
    (10007, 1, False, 4), (10007, 9, False, 4), (10007, 32, False, 4), (10007, 33, False, 4), (10007, 64, False, 4),
    (10007, 65, False, 0), (5003, 7, True, 4), (5003, 33, True, 2), (5003, 64, True, 2), (5003, 65, True, 0),
    (15013, 31, False, 4), (15013, 33, False, 2), (7919, 39, True, 2)])
def test_split_counts(gpu, n, batch, dbl, split):
    t, dt = (ff.Type.Z2Z, np.complex128) if dbl else (ff.Type.C2C, np.complex64)
    x = complex_input(n + batch, (batch, n), dt)
    xd = dev_tensor(x, gpu)
    yd, zd = dev_tensor(np.full_like(x, 7.0), gpu), dev_tensor(np.full_like(x, 7.0), gpu)
    with ff.Plan.one_d(n, t, batch) as p:
        p.set_stream(stream_of(gpu))
        word = f"k_bluestein_combine<fp{64 if dbl else 32},{split}>"
        assert (word in p.description()) if split else ("k_bluestein_ip" in p.description()), p.description()
        go = p.z2z if dbl else p.c2c
        go(xd.data_ptr(), yd.data_ptr(), ff.FORWARD)
        go(xd.data_ptr(), zd.data_ptr(), ff.INVERSE)
        sync(gpu)
    x64 = x.astype(np.complex128)
    check_accuracy(host(yd), np.fft.fft(x64, axis=1), t, n, row_len=n, what="fwd")
    check_accuracy(host(zd), np.fft.ifft(x64, axis=1) * n, t, n, row_len=n, what="inv")
