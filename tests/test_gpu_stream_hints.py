"""Large inputs are read, and outputs written, with non-temporal accesses (GPU).

A batch past the size where the hints start gives the same bits as its two
halves below it (which run on the same instances); the strides where a hint has to stay off (short or unaligned rows)
are among the lengths.  Parts are checked against the oracle elsewhere.
"""
import numpy as np
import pytest

from flagfft_amd import flagfft as ff

from .helpers import stream_of, sync

pytestmark = pytest.mark.gpu

CASES = [(1024, 16384, "c2c"), (1000, 17000, "c2c"), (64, 1 << 18, "c2c"), (1 << 20, 16, "c2c"), (65536, 256, "c2c"),
         (4096, 8192, "r2c"), (4096, 8192, "c2r"), (1 << 19, 64, "r2c"), (1 << 19, 64, "c2r"), (2048, 4096, "z2z"),
         (1 << 17, 64, "z2z")]


@pytest.mark.parametrize("n,batch,kind", CASES)
def test_large_batch_equals_its_parts(gpu, n, batch, kind):
    import torch

    dbl = kind == "z2z"
    cdt = torch.complex128 if dbl else torch.complex64
    h = n // 2 + 1
    t = {"c2c": ff.Type.C2C, "z2z": ff.Type.Z2Z, "r2c": ff.Type.R2C, "c2r": ff.Type.C2R}[kind]
    g = torch.Generator(device=gpu)
    g.manual_seed(n + batch)
    ni, dti = {"r2c": (n, torch.float32), "c2r": (h, cdt)}.get(kind, (n, cdt))
    no, dto = {"r2c": (h, cdt), "c2r": (n, torch.float32)}.get(kind, (n, cdt))
    x = torch.randn((batch, ni), dtype=dti, device=gpu, generator=g)
    outs = []
    for parts in (1, 2):
        b = batch // parts
        y = torch.empty((batch, no), dtype=dto, device=gpu)
        with ff.Plan.one_d(n, t, b) as p:
            p.set_stream(stream_of(gpu))
            for k in range(parts):
                i, o = x[k * b].data_ptr(), y[k * b].data_ptr()
                {"c2c": lambda: p.c2c(i, o), "z2z": lambda: p.z2z(i, o), "r2c": lambda: p.r2c(i, o),
                 "c2r": lambda: p.c2r(i, o)}[kind]()
            sync(gpu)
        outs.append(y)
    assert torch.equal(torch.view_as_real(outs[0]) if no != n or dto.is_complex else outs[0],
                       torch.view_as_real(outs[1]) if no != n or dto.is_complex else outs[1])
    assert bool(torch.isfinite(outs[0][:, :1].abs()).all()) and float(outs[0][-1].abs().sum()) > 0
