"""The kick that finalises its runs itself (up to 256 workgroups of 256 particles) against the separate
finalising launch (more): a run alone takes the first, batched with a large run the second. State, times,
time steps and conserved sums are equal bit for bit, through the priming step, steps and a reduction outside
a step, for one particle, one workgroup, a remainder of one, and the largest size that takes the first.
"""
from __future__ import annotations

import numpy as np
import pytest

from spearhed_amd import ic
from spearhed_amd.particles import ParticleSet
from spearhed_amd.stepper import Context


def _run(n):
    cfg, base = ic.mhd_turbulence(n=max(4, int(np.ceil(n ** (1.0 / 3.0)))), seed=n)
    pick = np.sort(np.random.default_rng(n).permutation(base.n)[:n])
    ps = ParticleSet(n)
    for name in ("id", "mask", "species", "mass", "rho", "h", "u", "psi"):
        setattr(ps, name, getattr(base, name)[pick])
    for name in ("pos", "vel", "B"):
        setattr(ps, name, getattr(base, name)[:, pick])
    return cfg, ps


def _result(runs, precision):
    with Context([c for c, _ in runs], [p.n for _, p in runs], precision=precision) as ctx:
        for r, (_, p) in enumerate(runs):
            ctx.upload(r, p)
        ctx.step(3)  # primes, then two steps
        sums = ctx.conserved()[0]
        ctx.step(1)
        return ctx.download(0), sums, ctx.conserved()[0]


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["mixed", "fp32"])
@pytest.mark.parametrize("n", [1, 256, 257, 4001, 65536])
def test_kick_finalizes_like_the_separate_launch(n, precision):
    print(f"n {n} {precision}", flush=True)
    own = _run(n)
    a, sums_a, end_a = _result([own], precision)
    b, sums_b, end_b = _result([own, _run(65600)], precision)
    for name in ("id", "pos", "vel", "u", "rho", "B", "psi", "dvdt", "vsig"):
        assert np.array_equal(getattr(a, name), getattr(b, name)), name
    assert sums_a == sums_b and end_a == end_b
