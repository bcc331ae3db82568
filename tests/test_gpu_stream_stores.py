"""Hinted and plain stores of the same transforms write the same bits (GPU).

A batch on one side of a hint's size line against its parts on the other (which run
on the same instances); the plans name the hints they run with.  Values are checked
against the oracle elsewhere.
"""
import pytest

from flagfft_amd import flagfft as ff

from .helpers import stream_of, sync

pytestmark = pytest.mark.gpu

# (kind, n, whole batch, parts, hint of the whole, hint of a part)
ROWS = [("c2c", 4096, 1536, 2, False, True), ("c2c", 1024, 6144, 2, False, True), ("z2z", 1024, 3072, 2, False, True),
        ("c2r", 4096, 3072, 2, False, True), ("r2c", 4096, 3072, 2, False, True), ("r2c", 2048, 256, 2, True, False),
        ("r2c", 1024, 6000, 2, False, True), ("d2z", 512, 6000, 2, False, True), ("d2z", 2048, 2560, 2, False, True),
        ("r2c", 1000, 4000, 2, False, False), ("r2c", 8, 300001, 1, False, False)]


@pytest.mark.parametrize("kind,n,batch,parts,whole,part", ROWS)
def test_rows(gpu, kind, n, batch, parts, whole, part):
    _compare(gpu, kind, n, batch, parts, whole, part)


# the split-spectrum pass of its own, lines at 32 MiB
POST = [("r2c", 752, 20000, 2, True, False), ("d2z", 1502, 5000, 2, True, False), ("r2c", 200000, 60, 2, True, False)]


@pytest.mark.parametrize("kind,n,batch,parts,whole,part", POST)
def test_split_spectrum_pass(gpu, kind, n, batch, parts, whole, part):
    _compare(gpu, kind, n, batch, parts, whole, part)


def _compare(gpu, kind, n, batch, parts, whole, part):
    import torch

    dbl = kind in ("z2z", "d2z")
    rdt, cdt = (torch.float64, torch.complex128) if dbl else (torch.float32, torch.complex64)
    h = n // 2 + 1
    t = ff.Type[kind.upper()]
    ni, dti = {"r2c": (n, rdt), "d2z": (n, rdt), "c2r": (h, cdt)}.get(kind, (n, cdt))
    no, dto = {"r2c": (h, cdt), "d2z": (h, cdt), "c2r": (n, rdt)}.get(kind, (n, cdt))
    g = torch.Generator(device=gpu)
    g.manual_seed(n + batch)
    x = torch.randn((batch, ni), dtype=dti, device=gpu, generator=g)
    outs = []
    for k, hint in ((1, whole), (parts, part)):
        b = batch // k
        y = torch.full((batch + 1, no), 7.0, dtype=dto, device=gpu)  # one row past the output
        with ff.Plan.one_d(n, t, b) as p:
            p.set_stream(stream_of(gpu))
            assert ("stream-out" in p.description()) == hint, p.description()
            for j in range(k):
                i, o = x[j * b].data_ptr(), y[j * b].data_ptr()
                if kind in ("c2c", "z2z"):
                    getattr(p, kind)(i, o, ff.FORWARD)
                else:
                    getattr(p, kind)(i, o)
            sync(gpu)
        assert bool((y[batch] == 7.0).all())
        outs.append(y[:batch] if not dto.is_complex else torch.view_as_real(y[:batch]))
    assert torch.equal(*outs) and bool(torch.isfinite(outs[0]).all()) and float(outs[0][-1].abs().sum()) > 0
