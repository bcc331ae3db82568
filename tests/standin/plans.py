"""Plans on the CPU stand-in runtime (hip_standin.cpp): run(queries) answers in a
process of its own with the stand-in preloaded.

A query is a dict: type, n (a list), batch, and optionally tuning (set_tuning's
keywords), limit (bytes of device memory), or server (arena bytes: submit one
request of n[0] x batch).  The answer holds the result code and, of a plan, its
launches as (label, stream-in, stream-out) per direction, its workspace and
table bytes, and the result codes of flagfftxExecC2CNoAlloc.
"""
from __future__ import annotations

import ctypes
import json
import os
import re
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))


def build(folder) -> str:
    so = os.path.join(str(folder), "hip_standin.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include",
                    "-Wno-attributes", os.path.join(HERE, "hip_standin.cpp"), "-o", so], check=True)
    return so


def run(so: str, queries: list[dict], env: dict | None = None) -> list[dict]:
    pre = os.environ.get("LD_PRELOAD")
    e = {**os.environ, "LD_PRELOAD": so + (":" + pre if pre else ""), "HIP_STANDIN": so, "FLAGFFT_TUNE_DISABLE": "1",
         **(env or {})}
    out = subprocess.run([sys.executable, os.path.abspath(__file__)], input=json.dumps(queries), text=True, cwd=ROOT,
                         env=e, stdout=subprocess.PIPE, stderr=subprocess.PIPE, timeout=600)
    assert out.returncode == 0, out.stderr[-2000:]
    return json.loads(out.stdout)


def launches(desc: str) -> list[list]:
    """[(label, stream-in, stream-out)] of each execution section of a description."""
    res = []
    for part in re.split(r"\n-- (?:Forward|Inverse) execution", desc)[1:]:
        lines = [l for l in part.split("\n") if l.startswith("  [")]
        if lines:
            res.append([(l.strip(), " stream-in" in l, " stream-out" in l) for l in lines])
    return res


def _answer(ff, st, q: dict) -> dict:
    t = ff.Type[q["type"]]
    n, batch = q["n"], q.get("batch", 1)
    limit = ctypes.c_longlong.in_dll(st, "standin_limit")
    live = ctypes.c_longlong.in_dll(st, "standin_live")
    if "server" in q:
        with ff.Server(q["server"], mode=ff.SERVE_PLAIN) as s:
            tk = ctypes.c_longlong()
            r = ff.lib().flagfftxServerSubmit(s.handle, int(t), n[0], batch, ff.FORWARD, 0x1000, ctypes.byref(tk))
            if r == 0:
                s.wait(tk.value)
        return {"result": r}
    if q.get("tuning"):
        ff.set_tuning(**q["tuning"])
    before = live.value
    limit.value = q.get("limit", 0)
    try:
        r, h = {1: lambda: ff.plan1d(n[0], t, batch), 2: lambda: ff.plan2d(n[0], n[1], t),
                3: lambda: ff.plan3d_ext(*n, t, batch)}[len(n)]()
    finally:
        limit.value = 0
        ff.set_tuning()
    a = {"result": int(r)}
    if r == 0:
        a["text"] = ff.description(h)
        a["launches"] = launches(a["text"])
        a["bytes"] = live.value - before
        if t == ff.Type.C2C:
            a["noalloc"] = [int(ff.exec_c2c_noalloc(h, 0x1000, 0x2000, d)) for d in (ff.FORWARD, ff.INVERSE)]
        ff.destroy(h)
    return a


if __name__ == "__main__":
    sys.path.insert(0, ROOT)
    from flagfft_amd import flagfft as lib_

    standin = ctypes.CDLL(os.environ["HIP_STANDIN"])
    print(json.dumps([_answer(lib_, standin, q) for q in json.load(sys.stdin)]))
