"""Asynchronous downloads: every column equals the synchronous download's, bit for bit.

A response to pinned memory is written by a kernel up to a size (by all XCDs up to 1 MiB, by one beyond), by
copies beyond it and to ordinary memory; a pool's goes through its ring. The cases hold one element, column
lengths that fill no vector, a second run whose columns start off any vector boundary, destinations at such a
start, and sizes on both sides of the change of kernel and of the limits (12 MiB in a context, 16 MiB out of
a pool's ring) at 78 bytes per particle.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from spearhed_amd import capi, ic
from spearhed_amd.particles import ParticleSet
from spearhed_amd.stepper import RESPONSE_FIELDS, Context, PinnedRing, Pool

FIELDS = ["id", "mask", "species", "pos", "vel", "mass", "rho", "h", "u", "B", "psi"]


def _run(n, seed):
    cfg, base = ic.mhd_turbulence(n=8, seed=seed)
    rng = np.random.default_rng(seed)
    ps = ParticleSet(n)
    ps.id = rng.permutation(n).astype(np.uint64)
    ps.pos = rng.uniform(0.0, 1.0, (3, n))
    for name in ("mass", "h", "u", "rho"):
        setattr(ps, name, np.full(n, getattr(base, name)[0], dtype=np.float32))
    ps.vel = rng.normal(0, 0.1, (3, n)).astype(np.float32)
    ps.B = rng.normal(0, 0.1, (3, n)).astype(np.float32)
    return cfg, ps


def _columns(n, ring, shift):
    """A response of n particles, each column `shift` elements into its buffer (the ring's, or ordinary memory)."""
    soa, out = capi.HostSoA(), {}
    soa.n = n
    for f in FIELDS:
        attr, dtype, comps = RESPONSE_FIELDS[f]
        cols = []
        for a in range(comps):
            col = (ring.take(dtype, n + shift) if ring else np.zeros(n + shift, dtype))[shift:]
            ptr = C.cast(col.ctypes.data, C.POINTER(np.ctypeslib.as_ctypes_type(dtype)))
            if comps > 1:
                getattr(soa, attr)[a] = ptr
            else:
                setattr(soa, attr, ptr)
            cols.append(col)
        out[f] = cols
    return soa, out


@pytest.mark.gpu
@pytest.mark.parametrize("pool", [False, True])
@pytest.mark.parametrize("pinned", [True, False])
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("n", [1, 63, 1001, 13000, 14500, 29001, 105000, 155000, 170001, 210000, 220001])
def test_download_async_equals_download(n, shift, pinned, pool):
    runs = [_run(257, 3), _run(n, 4)]
    total = sum(p.n for _, p in runs)
    if pool:
        cells = sum(int(capi.load().sph_run_cells(C.byref(c))) for c, _ in runs)
        ctx = Pool(5 * total, 2 * cells, 4, precision="mixed")
        ctx.set_runs([], [(c, p.n) for c, p in runs])
    else:
        ctx = Context([c for c, _ in runs], [p.n for _, p in runs], precision="mixed")
    print(f"n {n} shift {shift} pinned {pinned} pool {pool}", flush=True)
    ring = PinnedRing(128 * total + (1 << 16)) if pinned else None
    with ctx:
        for r, (_, p) in enumerate(runs):
            ctx.upload(r, p)
        ctx.resort()
        for r in (0, 1):
            soa, out = _columns(runs[r][1].n, ring, shift)
            capi.check(ctx.lib.sph_download_async(ctx.h, r, C.byref(soa), None), ctx.h, "sph_download_async")
            ctx.sync()
            want = ctx.download(r)
            for f in FIELDS:
                for a, col in enumerate(out[f]):
                    ref = np.asarray(getattr(want, f))
                    assert np.array_equal(col, ref[a] if ref.ndim > 1 else ref), f
    if ring:
        ring.close()
