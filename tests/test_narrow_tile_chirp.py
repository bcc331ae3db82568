"""Chirp sources and sinks on the narrow LDS tiles (729, 100, 125 and 1000 points): the
tiles that few units take (CPU), and their results (GPU).
"""
import re

import numpy as np
import pytest

from flagfft_amd import flagfft as ff

from .helpers import check_accuracy, complex_input, dev_tensor, host, stream_of, sync
from .standin import plans

# (type, n, batch, split, units per workgroup of the outer passes)
CASES = [("C2C", 31991, 1, [1000, 64], 4), ("C2C", 31991, 3, [1000, 64], 4), ("Z2Z", 31991, 1, [1000, 64], 4),
         ("C2C", 93307, 1, [729, 256], 4), ("C2C", 15991, 2, [125, 256], 8), ("Z2Z", 15991, 1, [125, 256], 8),
         ("C2C", 12799, 1, [100, 256], 8), ("Z2Z", 12799, 2, [100, 256], 8)]


def _outer_units(text):
    """Units per workgroup of the outer passes' launches."""
    got = re.findall(r"k_stage<fp\d\d,\d+,(\d+),0>", text.split("-- Inverse")[0])
    assert len(got) == 2, text
    return [int(u) for u in got]


@pytest.fixture(scope="module")
def described(tmp_path_factory):
    so = plans.build(tmp_path_factory.mktemp("standin"))
    got = plans.run(so, [{"type": t, "n": [n], "batch": b, "tuning": {"passes": s}} for t, n, b, s, _ in CASES])
    return [a["text"] for a in got]


@pytest.mark.parametrize("i", range(len(CASES)))
def test_few_units_take_the_narrow_tile(described, i):
    assert _outer_units(described[i]) == [CASES[i][4]] * 2


@pytest.mark.gpu
@pytest.mark.parametrize("t,n,batch,split,units", CASES)
def test_results(gpu, t, n, batch, split, units):
    ty = ff.Type[t]
    dt = np.complex64 if t == "C2C" else np.complex128
    x = complex_input(n + batch, (batch, n), dt)
    xd = dev_tensor(x, gpu)
    # (room past the result, which has to stay as it is)
    yd = dev_tensor(np.full(batch * n + 65536, 7.0, dt), gpu)
    ff.set_tuning(passes=split)
    try:
        p = ff.Plan.one_d(n, ty, batch)
    finally:
        ff.set_tuning()
    with p:
        assert _outer_units(p.description()) == [units] * 2
        p.set_stream(stream_of(gpu))
        for sign in (ff.FORWARD, ff.INVERSE):
            (p.c2c if t == "C2C" else p.z2z)(xd.data_ptr(), yd.data_ptr(), sign)
            sync(gpu)
            y, x64 = host(yd), x.astype(np.complex128)
            assert (y[batch * n:] == 7.0).all()
            ref = np.fft.fft(x64, axis=1) if sign == ff.FORWARD else np.fft.ifft(x64, axis=1) * n
            check_accuracy(y[:batch * n].reshape(batch, n), ref, ty, n, row_len=n, what=f"{split} {sign}")
