"""Odd real lengths whose convolution has 2048-point outer passes, with few sequences:
three launches on register-resident instances (CPU), as with many, and their results
(GPU).  The complex transforms of these lengths keep the LDS super-stage.
"""
import numpy as np
import pytest

from flagfft_amd import flagfft as ff

from .helpers import check_accuracy, complex_input, dev_tensor, host, real_input, stream_of, sync
from .standin import plans

CASES = [(1000003, 1), (600011, 1), (600011, 2), (160001, 8), (160001, 30), (135001, 3)]


@pytest.fixture(scope="module")
def described(tmp_path_factory):
    so = plans.build(tmp_path_factory.mktemp("standin"))
    keys = [(t, n, b) for t in ("R2C", "C2R", "C2C") for n, b in CASES]
    got = plans.run(so, [{"type": t, "n": [n], "batch": b} for t, n, b in keys])
    return {k: [l for l, _, _ in a["launches"][0]] for k, a in zip(keys, got)}


@pytest.mark.parametrize("n,batch", CASES)
@pytest.mark.parametrize("t", ["R2C", "C2R"])
def test_three_launches(described, t, n, batch):
    steps = described[(t, n, batch)]
    assert len(steps) == 3 and not any("k_pass" in s for s in steps), steps
    for s in (steps[0], steps[2]):
        assert "k_col<fp32" in s and "R=2048" in s, s


@pytest.mark.parametrize("n,batch", [c for c in CASES if c != (160001, 30)])
def test_few_complex_sequences_keep_the_super_stage(described, n, batch):
    steps = described[("C2C", n, batch)]
    assert len(steps) == 3 and all("k_stage" in s for s in (steps[0], steps[2])), steps


@pytest.mark.gpu
@pytest.mark.parametrize("n,batch", CASES)
def test_results(gpu, n, batch):
    h = n // 2 + 1
    x, Y = real_input(n, (batch, n), np.float32), complex_input(n + 1, (batch, h), np.complex64)
    xd, Yd = dev_tensor(x, gpu), dev_tensor(Y, gpu)
    # (room past each result, which has to stay as it is)
    Xd = dev_tensor(np.full(batch * h + 4096, 7.0, np.complex64), gpu)
    yd = dev_tensor(np.full(batch * n + 4096, 7.0, np.float32), gpu)
    with ff.Plan.one_d(n, ff.Type.R2C, batch) as pf, ff.Plan.one_d(n, ff.Type.C2R, batch) as pi:
        for p in (pf, pi):
            p.set_stream(stream_of(gpu))
        pf.r2c(xd.data_ptr(), Xd.data_ptr())
        pi.c2r(Yd.data_ptr(), yd.data_ptr())
        sync(gpu)
    X, y = host(Xd), host(yd)
    assert (X[batch * h:] == 7.0).all() and (y[batch * n:] == 7.0).all()
    check_accuracy(X[:batch * h].reshape(batch, h), np.fft.rfft(x.astype(np.float64), axis=1), ff.Type.R2C, n,
                   row_len=h, what="R2C")
    Y64 = Y.astype(np.complex128)
    Y64[:, 0] = Y64[:, 0].real  # Im of the DC bin does not count
    check_accuracy(y[:batch * n].reshape(batch, n), np.fft.irfft(Y64, n, axis=1) * n, ff.Type.C2R, n, row_len=n,
                   what="C2R")
