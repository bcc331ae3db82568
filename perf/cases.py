"""Transforms that programs run through the C ABI of this library, one per case.

A case is one plan (or the forward / inverse plan pair of a real transform)
and one pass over it: what a program that keeps its plan executes for one new
batch of data.  Fields:

shape      lengths of one transform, "4096" or "4096x4096" or "256x256x256"
           (row-major, the last axis contiguous)
batch      contiguous transforms of one execution (1D; 1 otherwise)
real       real <-> half-spectrum transforms (R2C / C2R, D2Z / Z2D)
double     FP64 instead of FP32
op         "forward", "inverse" or "roundtrip" (forward, then inverse of its
           output)
compute    arithmetic mode of 1024-point complex FP32 rows: 0 vector, 1 / 2
           BF16 / FP16 hi + lo on the matrix cores
"""
from __future__ import annotations

import math

import torch

from flagfft_amd import flagfft as ff


def _case(shape, batch=1, real=False, double=False, op="forward", compute=0, name=None):
    c = {"shape": shape, "batch": batch, "real": real, "double": double, "op": op, "compute": compute}
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest calls: a handful of short signals, filtered in the frequency domain
        _case("256", 4, op="roundtrip", name="signals_256x4"),
        # frames of a spectrogram or of overlap-add filtering
        _case("4096", 256, op="roundtrip", name="frames_4096x256"),
        # channel / range-line processing, the largest batch of short rows
        _case("1024", 65536, name="rows_1024x65536"),
        # one very long record
        _case("16777216", 1, name="record_2e24"),
        # long real records: spectrum and back
        _case("1048576", 16, real=True, op="roundtrip", name="real_records_2e20x16"),
        # filtering of one large image
        _case("4096x4096", real=True, op="roundtrip", name="image_4096"),
        # FP64 spectral solver, one field
        _case("2048x2048", double=True, name="field_f64_2048"),
        # volume of real samples: spectrum and back
        _case("256x256x256", real=True, op="roundtrip", name="volume_256"),
        # awkward lengths: a batch of prime-length sequences
        _case("10007", 64, name="prime_10007x64"),
        # long prime-length records, inverse direction
        _case("1000003", 4, op="inverse", name="prime_1000003x4"),
        # FP64 real frames of a decimal length
        _case("6000", 128, real=True, double=True, op="roundtrip", name="frames_f64_6000x128"),
        # an image of a decimal size
        _case("1000x1000", name="image_1000"),
    ]


# ---- more cases of the same ranges ----------------------------------------
def _log_uniform(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def _smooth(n):
    for p in (2, 3, 5, 7):
        while n % p == 0:
            n //= p
    return n == 1


def _length(rng, lo, hi):
    """A length in [lo, hi]: power of two, 7-smooth, or any integer (two, two and one of five)."""
    v = _log_uniform(rng, lo, hi)
    u = rng.random()
    if u < 0.4:
        return max(lo, min(hi, 1 << round(math.log2(v))))
    n = int(v)
    if u < 0.8:
        while not _smooth(n) and n > lo:
            n -= 1
    return max(n, lo)


def _drawn(rng):
    double = rng.random() < 0.25
    real = rng.random() < 0.4
    op = rng.choice(["forward", "inverse", "roundtrip"])
    u = rng.random()
    if u < 0.05:  # 1024-point rows on the matrix cores
        return _case("1024", int(_log_uniform(rng, 4, 65536)), op=op, compute=rng.choice([1, 2]))
    if u < 0.40:  # batches of short rows
        n = _length(rng, 32, 16384)
        batch = max(1, int(_log_uniform(rng, 1 << 10, 1 << 24) / n))
    elif u < 0.65:  # long records
        n = _length(rng, 16384, 1 << 22)
        batch = max(1, int(_log_uniform(rng, 1 << 16, 1 << 24) / n))
    elif u < 0.87:  # images and fields
        n0, n1 = _length(rng, 64, 4096), _length(rng, 64, 4096)
        return _case(f"{n0}x{n1}", real=real, double=double, op=op)
    else:  # volumes
        n0, n1, n2 = (_length(rng, 16, 256) for _ in range(3))
        return _case(f"{n0}x{n1}x{n2}", real=real, double=double, op=op)
    return _case(str(n), batch, real=real, double=double, op=op)


def draw(rng):
    """A case no larger than the listed ones: lengths that run as convolutions
    cost several times the others per sample, and more so along a strided axis."""
    while True:
        c = _drawn(rng)
        d = _dims(c)
        limit = 1 << 28
        if not all(_smooth(n) for n in d):
            limit = 1 << 26 if len(d) == 1 else 1 << 23
        if work(c)["bytes"] <= limit:
            return c


# ---- one case ---------------------------------------------------------------
def _dims(case):
    return tuple(int(s) for s in case["shape"].split("x"))


def _full_shape(case):
    d = _dims(case)
    return (case["batch"],) + d if len(d) == 1 else d


def _half_shape(case):
    s = _full_shape(case)
    return s[:-1] + (s[-1] // 2 + 1,)


def _axes(case):
    return tuple(range(-len(_dims(case)), 0))


def _input(case, seed, device):
    """N(0, 1) samples (re and im each), or the half spectrum of real ones."""
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    rdt = torch.float64 if case["double"] else torch.float32
    if not case["real"]:
        x = torch.randn(_full_shape(case) + (2,), dtype=rdt, device=device, generator=g)
        return torch.view_as_complex(x)
    if case["op"] != "inverse":
        return torch.randn(_full_shape(case), dtype=rdt, device=device, generator=g)
    # a half spectrum that some real signal has: bins that are their own
    # mirror image along the last axis come from real transforms
    n = _dims(case)[-1]
    lead, m = _full_shape(case)[:-1], n // 2 + 1
    z = torch.view_as_complex(torch.randn(lead + (m, 2), dtype=rdt, device=device, generator=g))
    axes = tuple(a for a in _axes(case) if a != -1)
    own = [0] + ([m - 1] if n % 2 == 0 else [])
    for k in own:
        if not axes:
            z[..., k].imag = 0
            continue
        col = z[..., k]
        mirror = col
        for a in range(col.dim()):
            mirror = torch.roll(torch.flip(mirror, (a,)), 1, a)
        z[..., k] = (col + mirror.conj()) / 2
    return z


def _plan(case, type_):
    d = _dims(case)
    if case["compute"]:
        return ff.Plan.one_d_compute(d[0], type_, case["batch"], case["compute"])
    if len(d) == 1:
        return ff.Plan.one_d(d[0], type_, case["batch"])
    if len(d) == 2:
        return ff.Plan.two_d(d[0], d[1], type_)
    return ff.Plan.three_d(d[0], d[1], d[2], type_)


def prepare(case, seed):
    dev = torch.device("cuda")
    T = ff.Type
    fwd_t, inv_t = (T.D2Z, T.Z2D) if case["double"] else (T.R2C, T.C2R)
    if not case["real"]:
        fwd_t = inv_t = T.Z2Z if case["double"] else T.C2C
    cdt = torch.complex128 if case["double"] else torch.complex64
    rdt = torch.float64 if case["double"] else torch.float32
    state = {"case": case, "x": _input(case, seed, dev)}
    stream = torch.cuda.current_stream().cuda_stream
    if case["op"] != "inverse":
        state["fwd"] = _plan(case, fwd_t)
        state["fwd"].set_stream(stream)
        state["spec"] = torch.empty(_half_shape(case) if case["real"] else _full_shape(case), dtype=cdt, device=dev)
    if case["op"] != "forward":
        same = "fwd" in state and not case["real"]  # a complex plan runs both directions
        state["inv"] = state["fwd"] if same else _plan(case, inv_t)
        state["inv"].set_stream(stream)
        state["back"] = torch.empty(_full_shape(case), dtype=rdt if case["real"] else cdt, device=dev)
    return state


def run(state):
    case = state["case"]
    src = state["x"]
    out = []
    if "fwd" in state:
        p, dst = state["fwd"], state["spec"]
        if case["real"]:
            (p.d2z if case["double"] else p.r2c)(src.data_ptr(), dst.data_ptr())
        else:
            (p.z2z if case["double"] else p.c2c)(src.data_ptr(), dst.data_ptr(), ff.FORWARD)
        out.append(dst)
        src = dst
    if "inv" in state:
        p, dst = state["inv"], state["back"]
        if case["real"]:
            (p.z2d if case["double"] else p.c2r)(src.data_ptr(), dst.data_ptr())
        else:
            (p.z2z if case["double"] else p.c2c)(src.data_ptr(), dst.data_ptr(), ff.INVERSE)
        out.append(dst)
    return out


def exact(case, seed):
    """The unnormalised transforms in 64 bits on the host."""
    x = _input(case, seed, torch.device("cuda")).cpu()
    x = x.to(torch.complex128 if x.is_complex() else torch.float64)
    ax = _axes(case)
    d = _dims(case)
    out = []
    if case["op"] != "inverse":
        spec = torch.fft.rfftn(x, dim=ax) if case["real"] else torch.fft.fftn(x, dim=ax)
        out.append(spec)
        if case["op"] == "roundtrip":
            out.append(x * float(math.prod(d)))
    elif case["real"]:
        out.append(torch.fft.irfftn(x, s=d, dim=ax, norm="forward"))
    else:
        out.append(torch.fft.ifftn(x, dim=ax, norm="forward"))
    return out


def work(case):
    """Input read once, output written once per execution; 5 n log2 n operations of a
    complex n-point transform, half of that of a real one."""
    eb = 16 if case["double"] else 8
    total = math.prod(_full_shape(case))
    n = math.prod(_dims(case))
    if case["real"]:
        nbytes = total * eb // 2 + math.prod(_half_shape(case)) * eb
    else:
        nbytes = 2 * total * eb
    flops = 5.0 * total * math.log2(n) * (0.5 if case["real"] else 1.0)
    execs = 2 if case["op"] == "roundtrip" else 1
    return {"bytes": nbytes * execs, "flops": flops * execs}
