"""Which launches of a plan carry cache hints (CPU: plans on the stand-in runtime).

Non-temporal loads: inputs of 128 MiB and more whose accesses are whole 128-byte
lines.  A line that several accesses share is fetched for each of them: 8- to
64-point rows ran up to 1.8 times longer with the hint.
"""
import pytest

from .standin import plans

MIB = 1 << 20


@pytest.fixture(scope="module")
def standin(tmp_path_factory):
    return plans.build(tmp_path_factory.mktemp("standin"))


def _launches(so, cases):
    """Per (type, n, batch): the launches of the plan's (forward) execution."""
    res = plans.run(so, [dict(type=t, n=list(n) if isinstance(n, tuple) else [n], batch=b) for t, n, b in cases])
    assert all(r["result"] == 0 for r in res)
    return [r["launches"][0] for r in res]


# (type, n, batch, the first launch's loads are hinted)
LOADS = [("C2C", 1024, 16384, True), ("C2C", 1024, 16383, False), ("C2C", 256, 1 << 17, True),
         # tpu threads read runs of 8 tpu bytes (FP32): 8 .. 64 points 8-32 bytes, 128 points 64, 1000 points 504
         ("C2C", 8, 1 << 22, False), ("C2C", 16, 1 << 21, False), ("C2C", 32, 1 << 20, False),
         ("C2C", 64, 1 << 19, False), ("C2C", 128, 1 << 18, False), ("C2C", 1000, 40000, False),
         ("Z2Z", 64, 1 << 18, False), ("Z2Z", 128, 1 << 17, True),
         ("R2C", 64, 1 << 21, False), ("R2C", 256, 1 << 19, False), ("R2C", 512, 1 << 17, True), ("D2Z", 256, 1 << 17, True),
         # half-spectrum rows of N + 1 bins are never whole lines
         ("C2R", 128, 1 << 19, False), ("C2R", 4096, 1 << 14, False), ("Z2D", 64, 1 << 19, False),
         # chains: the first pass, of R2C up to 224 MiB
         ("C2C", 1 << 20, 16, True), ("C2C", 1 << 20, 15, False), ("Z2Z", 1 << 20, 16, True), ("R2C", 1 << 20, 32, True),
         ("R2C", 1 << 20, 31, False), ("R2C", 1 << 20, 55, True), ("R2C", 1 << 20, 56, False), ("D2Z", 1 << 20, 27, True),
         ("D2Z", 1 << 20, 32, False), ("R2C", 1 << 25, 1, True), ("R2C", 1 << 25, 2, False), ("C2R", 1 << 20, 64, False),
         # the split-spectrum pass of its own ahead of a C2R chain, to 224 MiB as well
         ("C2R", 1 << 24, 2, True), ("C2R", 1502, 27924, True), ("C2R", 1502, 22000, False), ("C2R", 1502, 39200, False),
         ("Z2D", 1 << 23, 2, True), ("C2R", 1 << 24, 4, False),
         ("C2C", (4096, 4096), 1, True), ("R2C", (8192, 4096), 1, True), ("C2C", (256, 256, 256), 1, True)]


def test_loads(standin):
    for (t, n, b, want), steps in zip(LOADS, _launches(standin, [c[:3] for c in LOADS])):
        assert steps[0][1] == want, (t, n, b, steps)
        assert not any(s[1] for s in steps[1:]), (t, n, b, steps)


# (type, n, batch, the output's stores are hinted): rows up to 32 MiB in whole lines;
# half-spectrum rows from 2 MiB on in runs of 256 bytes, to 16 MiB or, with 48 threads
# a row, 32
STORES = [("C2C", 1024, 4096, True), ("C2C", 1024, 4097, False), ("C2C", 128, 4096, False), ("C2C", 256, 4096, True),
          ("C2C", 1000, 2000, False), ("C2R", 4096, 2048, True), ("C2R", 4096, 2049, False),
          ("R2C", 8, 300000, False), ("R2C", 32, 40000, False), ("R2C", 512, 8000, False), ("R2C", 1024, 4088, True),
          ("R2C", 1024, 4090, False), ("D2Z", 256, 6000, False), ("D2Z", 512, 3000, True), ("D2Z", 512, 4100, False),
          ("R2C", 1536, 2000, True), ("R2C", 2048, 256, True), ("R2C", 2048, 255, False),
          ("R2C", 2048, 4091, True), ("R2C", 2048, 4093, False), ("D2Z", 1536, 1000, True)]


def test_row_stores(standin):
    for (t, n, b, want), steps in zip(STORES, _launches(standin, [c[:3] for c in STORES])):
        assert len(steps) == 1 and steps[0][2] == want, (t, n, b, steps)


# the split-spectrum pass of its own: from 32 MiB on
POST = [("R2C", 752, 419, False), ("R2C", 752, 11100, False), ("R2C", 752, 11140, True), ("D2Z", 1502, 2780, False),
        ("D2Z", 1502, 2800, True), ("R2C", 1 << 25, 1, True)]


def test_split_spectrum_pass(standin):
    for (t, n, b, want), steps in zip(POST, _launches(standin, [c[:3] for c in POST])):
        assert "k_real_post" in steps[-1][0] and steps[-1][2] == want, (t, n, b, steps)
