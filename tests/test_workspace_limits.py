"""Convolution lengths against the limits on workspace (CPU: plans on the stand-in
runtime): the fixed scratch array of flagfftxExecC2CNoAlloc, a server's arena and
device memory.  The measure is the shortest product of two fast super-radices,
M >= 2 n - 1: what fits with it is accepted, though plans without a limit may take a
longer and faster M.
"""
import random

import pytest

from flagfft_amd import flagfft as ff

from .standin import plans

SCRATCH = 64 << 20
# power-of-two and 3-smooth super-radices of the compiled passes (FP32 and FP64)
FAST = [64, 81, 128, 135, 160, 256, 512, 729, 1024, 2048]


def shortest(n, largest=4096):
    fast = [r for r in FAST + [4096] if r <= largest]
    return min(a * b for a in fast for b in fast if a * b >= 2 * n - 1)


def two_workspaces(n, batch, elem=8):
    return 2 * ((batch * shortest(n) * elem + 255) // 256 * 256)


@pytest.fixture(scope="module")
def standin(tmp_path_factory):
    return plans.build(tmp_path_factory.mktemp("standin"))


def _cases():
    rng = random.Random(7)
    cases = [(26259, 69), (49133, 38), (24709, 69), (48513, 42), (48935, 35), (27307, 68), (54433, 34)]
    while len(cases) < 150:
        n = int(20300 * (2.0e6 / 20300) ** rng.random()) | 1
        batch = max(1, int(SCRATCH * rng.uniform(0.93, 1.05) / (16 * shortest(n))))
        if any(n % p == 0 for p in (3, 5, 7, 11, 13, 17, 19)):
            continue
        cases.append((n, batch))
    return cases


def test_scratch_array(standin):
    cases = _cases()
    res = plans.run(standin, [dict(type="C2C", n=[n], batch=b) for n, b in cases])
    held = 0
    for (n, b), r in zip(cases, res):
        assert r["result"] == 0 and "Bluestein" in r["text"], (n, b)
        if two_workspaces(n, b) <= SCRATCH:
            held += 1
            assert r["noalloc"] == [0, 0], (n, b, r["text"])
        else:
            assert r["noalloc"] == [ff.Result.INVALID_SIZE] * 2, (n, b)
    assert held > 60


@pytest.mark.parametrize("n,batch", [(48197, 16), (28001, 3), (53105, 20), (48197, 1)])
@pytest.mark.parametrize("t", ["C2C", "R2C"])
def test_server_arena(standin, t, n, batch):
    out = batch * n * 8 if t == "C2C" else batch * (n // 2 + 1) * 8
    fits = out + two_workspaces(n, batch) + 3 * 256
    res = plans.run(standin, [dict(type=t, n=[n], batch=batch, server=s) for s in (fits, 2 * fits, fits * 9 // 10)])
    assert [r["result"] for r in res] == [0, 0, ff.Result.ALLOC_FAILED]


def test_device_memory(standin):
    n, batch = 48197, 300
    (free,) = plans.run(standin, [dict(type="R2C", n=[n], batch=batch)])
    least = two_workspaces(n, batch)
    assert free["bytes"] > least * 1.3
    short, none = plans.run(standin, [dict(type="R2C", n=[n], batch=batch, limit=int(least * 1.1)),
                                      dict(type="R2C", n=[n], batch=batch, limit=int(least * 0.9))])
    assert short["result"] == 0 and short["bytes"] < least * 1.1 and "conv_length=98415" in short["text"]
    assert none["result"] == ff.Result.ALLOC_FAILED
