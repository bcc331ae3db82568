"""Queued register-resident passes give the bits of the same passes launched on their own,
for plain chains and for Bluestein chain ends, FP32 and FP64 instances of 16 to 64
elements per thread (GPU).
"""
import numpy as np
import pytest

from flagfft_amd import flagfft as ff

from .helpers import complex_input, d2h, dev_tensor, host, stream_of, sync

pytestmark = pytest.mark.gpu

# (n, batch, FP64, queued super-radices): 128 = 16 x 8, 64 = 8 x 8, 32 = 8 x 4, 16 = 4 x 4, 512 = 32 x 16,
# FP64 64 = 8 x 8
CHAINS = [(16384, 8, False, [128, 128]), (8192, 5, False, [128, 64]), (262144, 1, False, [512, 512]),
          (4096, 9, True, [64, 64])]


@pytest.mark.parametrize("n,batch,dbl,passes", CHAINS)
@pytest.mark.parametrize("sign", [ff.FORWARD, ff.INVERSE])
def test_same_bits_as_launched_alone(gpu, n, batch, dbl, passes, sign):
    t = ff.Type.Z2Z if dbl else ff.Type.C2C
    dt = np.complex128 if dbl else np.complex64
    x = complex_input(n + batch, (batch, n), dt)
    xd = dev_tensor(x, gpu)
    yd = xd.clone().zero_()
    ff.set_tuning(passes=passes)
    try:
        p = ff.Plan.one_d(n, t, batch)
    finally:
        ff.set_tuning()
    with p:
        assert p.description().count("k_col<") >= 2, p.description()
        p.set_stream(stream_of(gpu))
        (p.z2z if dbl else p.c2c)(xd.data_ptr(), yd.data_ptr(), sign)
        sync(gpu)
    with ff.Server(1 << 28) as srv:
        tk = srv.submit(t, n, batch, xd.data_ptr(), sign)
        ptr, _ = srv.wait(tk)
        got = d2h(ptr, (batch, n), dt)
        srv.release(tk)
        assert srv.stats()["queue_launches"] >= len(passes)
    assert np.array_equal(got, host(yd))
