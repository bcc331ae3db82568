"""Pass splits by the size of the whole transform: the splits measured fastest on both
sides of each line (CPU), and their results against the oracle (GPU).
"""
import re

import numpy as np
import pytest

from flagfft_amd import flagfft as ff
from oracle import oracle as ora

from .helpers import check_accuracy, complex_input, dev_tensor, host, stream_of, sync

# (type, n, batch, super-radices)
SPLITS = [("Z2Z", 262144, 1, [1024, 256]), ("Z2Z", 262144, 64, [1024, 256]), ("D2Z", 524288, 4, [1024, 256]),
          # the 4-unit tile counts to 24 MiB
          ("Z2Z", 150528, 6, [588, 256]), ("Z2Z", 150528, 13, [512, 294]), ("Z2Z", 3763200, 1, [160, 160, 147]),
          # run-time-radix passes of 512 to 1023 points past 64 MiB
          ("Z2Z", 294912, 7, [576, 512]), ("Z2Z", 294912, 28, [1152, 256]),
          # FP32 ones over 2048 points with more than 256 units, to 20 MiB
          ("C2C", 150528, 1, [2352, 64]), ("C2C", 150528, 4, [2352, 64]), ("C2C", 150528, 5, [512, 294]),
          ("C2C", 602112, 1, [2352, 256]), ("C2C", 291600, 1, [2160, 135]), ("C2C", 291600, 2, [2916, 100]), ("C2C", 150528, 13, [512, 294]), ("C2C", 291600, 7, [729, 400]),
          ("C2C", 602112, 13, [2352, 256])]


def _radices(t, n, batch):
    r, text = ff.describe_host(1, [n], ff.Type[t], batch)
    assert r == ff.Result.SUCCESS
    return [int(v) for v in re.search(r"super_radices=\[([\d,]+)\]", text).group(1).split(",")]


@pytest.mark.parametrize("t,n,batch,want", SPLITS)
def test_split(t, n, batch, want):
    assert _radices(t, n, batch) == want


@pytest.mark.parametrize("t", ["C2C", "Z2Z"])
def test_every_size_has_a_split_of_n(t):
    for n in (150528, 179200, 262144, 291600, 315000, 602112, 645120, 3763200):
        for batch in (1, 2, 5, 13, 40, 200):
            assert int(np.prod(_radices(t, n, batch))) == n


@pytest.mark.gpu
@pytest.mark.parametrize("t,n,batch", [("Z2Z", 150528, 6), ("Z2Z", 150528, 13), ("C2C", 150528, 1), ("C2C", 150528, 13),
                                       ("C2C", 291600, 7), ("Z2Z", 294912, 7)])
def test_both_sides(gpu, t, n, batch):
    dbl = t == "Z2Z"
    x = complex_input(n + batch, (batch, n), np.complex128 if dbl else np.complex64)
    xd = dev_tensor(x, gpu)
    yd = dev_tensor(np.full_like(x, 7.0), gpu)
    with ff.Plan.one_d(n, ff.Type[t], batch) as p:
        p.set_stream(stream_of(gpu))
        (p.z2z if dbl else p.c2c)(xd.data_ptr(), yd.data_ptr(), ff.FORWARD)
        sync(gpu)
    check_accuracy(host(yd), ora.fft(x.astype(np.complex128)), ff.Type[t], n, row_len=n, what=f"{t} {n} x {batch}")
