"""GPU pair passes against the oracle over the candidate lists a supercell can have (27-cell stencil).

Each case puts the same number of particles into most supercells, so that the lists take the sizes where
the kept-candidate filter and the equal chunks change course: one particle per supercell (64 lanes to it),
lane counts per target that are no power of two, a kept list just around the 96 entries held beside a
chunk and around multiples of a chunk, lists just below and above the filter's limit of 768 candidates,
and 64 and 65 targets (one and two groups). A third of the supercells of the "holes" variant is empty, so
the list's segments have gaps; "walls" has no periodic images, so border stencils are short; "two_h" takes
the kernels for unequal smoothing lengths.

Neighbour counts are exact. Density is a sum of positive terms, the particle's own the largest of them: at
most about 770 FP32 additions split over lanes, within the parity tests' 1e-5 of the oracle. A particle's
forces come from the same pairs in the same order whatever the chunk, so both force chunks give the same
bits; they are not held to the oracle here, because a target with one or two neighbours, both close to the
support radius, has forces as uncertain as 1 - r/H in FP32 (the parity tests hold full neighbourhoods).
"""
from __future__ import annotations

import numpy as np
import pytest

from parity import assert_scaled, gpu_stages, oracle_stages
from spearhed_amd import capi
from spearhed_amd.particles import ParticleSet

CELLS = (5, 4, 3)


def _case(per_cell: int, variant: str):
    rng = np.random.default_rng(1000 + per_cell)
    e = 0.25
    lo = []
    for c in np.ndindex(*CELLS):
        if variant == "holes" and (c[0] + 2 * c[1] + c[2]) % 3 == 0:
            continue
        lo.append(np.array(c, dtype=np.float64)[:, None] * e + rng.uniform(0.02 * e, 0.98 * e, (3, per_cell)))
    pos = np.concatenate(lo, axis=1)
    h0 = 0.49 * e
    ps = ParticleSet(pos.shape[1])
    ps.id = np.arange(ps.n, dtype=np.uint64)
    ps.pos = pos
    ps.mass = np.full(ps.n, e ** 3 / per_cell, dtype=np.float32)
    ps.h = np.full(ps.n, h0, dtype=np.float32)
    if variant == "two_h":
        ps.h[1::2] = np.float32(0.8 * h0)
    ps.u = np.full(ps.n, 1.5, dtype=np.float32)
    ps.rho = np.ones(ps.n, dtype=np.float32)
    ps.vel = rng.normal(0, 0.1, size=(3, ps.n)).astype(np.float32)
    ps.B = np.stack([np.full(ps.n, 0.1), rng.normal(0, 0.02, ps.n), np.zeros(ps.n)]).astype(np.float32)
    wall = variant == "walls"
    cfg = capi.make_config(box_len=tuple(n * e for n in CELLS), periodic=(0, 0, 0) if wall else (1, 1, 1),
                           kernel=capi.KERNEL_WENDLAND, h0=h0, mhd=1, cleaning=1, borve=1)
    return cfg, ps


@pytest.mark.gpu
@pytest.mark.parametrize("variant", ["full", "holes", "walls", "two_h"])
@pytest.mark.parametrize("per_cell", [1, 2, 3, 5, 6, 9, 11, 13, 21, 28, 29, 64, 65])
def test_pair_passes_over_list_sizes(per_cell, variant):
    cfg, ps = _case(per_cell, variant)
    print(f"per_cell {per_cell} {variant} n={ps.n}", flush=True)
    g, g128 = (gpu_stages(cfg, ps, "mixed", tuning=dict(density_chunk=128, force_chunk=fc)) for fc in (64, 128))
    o = oracle_stages(cfg, ps, "mixed", ("resort", "density"))
    order = o.by_id()
    assert np.array_equal(g.nnb, o.nnb[order]), "neighbour counts differ"
    assert_scaled(g.rho, o.rho[order], o.sc_rho[order], "density")
    for name in ("dvdt", "dudt", "dbdt", "divb", "dpsidt", "vsig"):
        assert np.array_equal(getattr(g, name), getattr(g128, name)), name


@pytest.mark.gpu
@pytest.mark.parametrize("per_cell", [1, 3, 13, 28, 29])
def test_mostly_empty_box_gives_the_same_forces(per_cell):
    """The same particles in a box of 36 times as many supercells of the same edge, nearly all empty: the force
    pass takes its loads in another order there, and the results keep their bits."""
    cfg, ps = _case(per_cell, "walls")
    g = gpu_stages(cfg, ps, "mixed")
    for a, cells in enumerate((40, 18, 3)):
        cfg.box_len[a] = cells * 0.25
    print(f"per_cell {per_cell} in a mostly empty box n={ps.n}", flush=True)
    w = gpu_stages(cfg, ps, "mixed")
    for name in ("rho", "nnb", "dvdt", "dudt", "dbdt", "divb", "dpsidt", "vsig"):
        assert np.array_equal(getattr(g, name), getattr(w, name)), name
