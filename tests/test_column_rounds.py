"""4096-point FP32 columns of several transforms whose columns the tiles do not divide: one
pass when its workgroups fill the CUs (CPU), and its results (GPU).
"""
import numpy as np
import pytest

from flagfft_amd import flagfft as ff

from .helpers import check_accuracy, complex_input, dev_tensor, host, real_input, stream_of, sync
from .standin import plans

N1 = 4096


# (n0, n2, type, one pass): 256 CUs, 8 columns per tile
CASES = [(8, 500, "R2C", True), (8, 251, "C2C", True), (16, 251, "C2C", True), (8, 256, "C2C", True),
         (6, 251, "C2C", False), (8, 258, "C2C", False)]


@pytest.fixture(scope="module")
def described(tmp_path_factory):
    so = plans.build(tmp_path_factory.mktemp("standin"))
    got = plans.run(so, [{"type": t, "n": [n0, N1, n2]} for n0, n2, t, _ in CASES])
    return {c: a["text"] for c, a in zip(CASES, got)}


@pytest.mark.parametrize("case", CASES)
def test_passes(described, case):
    axis1 = described[case].split("columns (axis 1):")[1].split("columns (axis 0):")[0]
    assert ("Leaf(n=4096" in axis1) == case[3], described[case]


@pytest.mark.gpu
@pytest.mark.parametrize("n0,n2", [(8, 251), (16, 125)])
def test_results_complex(gpu, n0, n2):
    x = complex_input(n0 + n2, (n0, N1, n2), np.complex64)
    xd = dev_tensor(x, gpu)
    yd = dev_tensor(np.full(x.size + 65536, 7.0, np.complex64), gpu)
    with ff.Plan.three_d(n0, N1, n2, ff.Type.C2C) as p:
        assert "R=4096" in p.description(), p.description()
        p.set_stream(stream_of(gpu))
        p.c2c(xd.data_ptr(), yd.data_ptr(), ff.FORWARD)
        sync(gpu)
    y = host(yd)
    assert (y[x.size:] == 7.0).all()
    check_accuracy(y[:x.size].reshape(x.shape), np.fft.fftn(x.astype(np.complex128)), ff.Type.C2C, x.size, row_len=x.size)


@pytest.mark.gpu
def test_results_real(gpu):
    n0, n2 = 8, 500
    h = n2 // 2 + 1
    x = real_input(n2, (n0, N1, n2), np.float32)
    xd = dev_tensor(x, gpu)
    yd = dev_tensor(np.full(n0 * N1 * h + 65536, 7.0, np.complex64), gpu)
    with ff.Plan.three_d(n0, N1, n2, ff.Type.R2C) as p:
        p.set_stream(stream_of(gpu))
        p.r2c(xd.data_ptr(), yd.data_ptr())
        sync(gpu)
    y = host(yd)
    assert (y[n0 * N1 * h:] == 7.0).all()
    check_accuracy(y[:n0 * N1 * h].reshape(n0, N1, h), np.fft.rfftn(x.astype(np.float64)), ff.Type.R2C, x.size,
                   row_len=n0 * N1 * h)
