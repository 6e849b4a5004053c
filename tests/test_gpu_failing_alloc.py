"""Queries whose optional buffers cannot be allocated: the ordered copy of the
resident set, the scratch it is made with, the ordered query frames.  The
runtime refuses one chosen allocation, and the query takes the route that does
without, with the same rows, not exact rows nor an error.  In a process of
its own, where failing_alloc.c stands in front of the runtime's calls."""
import ctypes
import json
import os
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
pytestmark = pytest.mark.gpu


def _shim(path):
    shim = ctypes.CDLL(path, mode=ctypes.RTLD_GLOBAL)
    shim.fail_alloc.argtypes = [ctypes.c_int, ctypes.c_long]
    shim.alloc_calls.restype = ctypes.c_long
    sys.path.insert(0, os.path.dirname(HERE))
    return shim


def say(name, **kw):
    print(json.dumps(dict(name=name, **kw)), flush=True)


def child_optional(shim):
    from mdsctk_amd import knn, synth
    n_ref, natoms, k, m = 8200, 520, 12, 4100
    x = synth.metastable_trajectory(n_ref + m, natoms, 3, n_centres=12)
    ref, fit, w = x[:n_ref], x[n_ref:], synth.masses(natoms, "random", 2)
    want = None
    # the second query of 4100 frames makes the ordered copy (8200 seen)
    for call in (-1, 0, 1, 2):
        print(f"call {call}, synchronous", flush=True)
        with knn.KnnContext(0, "bf16") as ctx:
            ctx.set_reference(ref, w)
            d0, i0 = ctx.query(fit, k)
            want = want or (d0, i0)
            for turn in (0, 1):
                shim.fail_alloc(0, call if turn == 0 else -1)
                d, i = ctx.query(fit, k)
                say("sync", call=call, turn=turn, allocs=shim.alloc_calls(0),
                    same=bool((d == want[0]).all() and (i == want[1]).all()),
                    fallback=ctx.stats()["n_fallback_rows"], text=ctx.last_error())
        print(f"call {call}, served", flush=True)
        with knn.KnnContext(0, "bf16") as ctx:
            ctx.set_reference(ref, w)
            ctx.query(fit, k)
            ctx.wait(ctx.submit(fit[:2048], k))
            ctx.wait(ctx.submit(fit[:1900], k))
            for turn in (0, 1):
                shim.fail_alloc(0, call if turn == 0 else -1)
                r = ctx.wait(ctx.submit(fit[:2048], k))
                say("served", call=call, turn=turn, allocs=shim.alloc_calls(0),
                    same=bool((r.dist == want[0][:2048]).all() and (r.idx == want[1][:2048]).all()),
                    fallback=r.info["n_fallback_rows"], text="")
    print("DONE", flush=True)


def child_retry(shim):
    """The copy is refused once, for its memory or because the free memory's
    size cannot be had, and made after as many frames more."""
    from mdsctk_amd import knn, synth
    n_ref, natoms, k, m = 8200, 520, 12, 4100
    x = synth.metastable_trajectory(n_ref + m, natoms, 3, n_centres=12)
    want = None
    for kind in (0, 2):
        print(f"kind {kind}", flush=True)
        with knn.KnnContext(0, "bf16") as ctx:
            ctx.set_reference(x[:n_ref])
            for turn in range(5):
                shim.fail_alloc(kind, 0 if turn == 1 else -1)
                shim.fail_alloc(2 - kind, -1)
                d, i = ctx.query(x[n_ref:], k)
                want = want or (d, i)
                say("retry", kind=kind, turn=turn, held=ctx.stats()["device_bytes"],
                    same=bool((d == want[0]).all() and (i == want[1]).all()),
                    fallback=ctx.stats()["n_fallback_rows"], copy=12 * n_ref * natoms)
    print("DONE", flush=True)


def child_pinned(shim):
    from mdsctk_amd import knn, synth
    x = synth.trajectory(500, 40, 1)
    want = None
    for call in (-1, 0):
        print(f"call {call}", flush=True)
        with knn.KnnContext(0, "bf16") as ctx:
            ctx.set_reference(x)
            for turn in (0, 1):
                shim.fail_alloc(1, call if turn == 0 else -1)
                d, i = ctx.query(None, 8)
                want = want or (d, i)
                say("pinned", call=call, turn=turn,
                    same=bool((d == want[0]).all() and (i == want[1]).all()))
    print("DONE", flush=True)


def _run(shim, name):
    p = subprocess.run([sys.executable, "-u", os.path.abspath(__file__), shim, name],
                       capture_output=True, text=True, timeout=100)
    print(p.stdout[-6000:], p.stderr[-3000:])
    assert p.returncode == 0 and "DONE" in p.stdout
    return [json.loads(l) for l in p.stdout.splitlines() if l.startswith("{")]


@pytest.fixture(scope="module")
def shim(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("shim") / "failing_alloc.so")
    subprocess.run(["cc", "-shared", "-fPIC", "-O1", "-o", lib,
                    os.path.join(HERE, "failing_alloc.c"), "-ldl"], check=True)
    return lib


def test_optional_buffers_that_cannot_be_allocated(shim):
    rows = _run(shim, "optional")
    assert len(rows) == 16
    for r in rows:
        assert r["same"] and r["fallback"] == 0 and r["text"] == "", r
    assert any(r["allocs"] >= 3 for r in rows if r["call"] == -1 and r["name"] == "sync")


def test_the_ordered_copy_is_asked_for_again(shim):
    rows = _run(shim, "retry")
    assert len(rows) == 10
    for r in rows:
        assert r["same"] and r["fallback"] == 0, r
        base = next(b["held"] for b in rows if b["kind"] == r["kind"] and b["turn"] == 0)
        made = r["held"] > base + r["copy"]
        assert made == (r["turn"] >= 3), r


def test_pinned_output_buffer_that_cannot_be_allocated(shim):
    rows = _run(shim, "pinned")
    assert len(rows) == 4 and all(r["same"] for r in rows), rows


if __name__ == "__main__":
    globals()["child_" + sys.argv[2]](_shim(sys.argv[1]))
