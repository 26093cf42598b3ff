"""Supercell starts and sort order against the oracle over supercell counts (exact).

The histogram is scanned whole by the scatter (up to 8,192 supercells), in blocks of 2,048 whose offsets the
scatter scans (up to 256 of them), or with the offsets scanned by a kernel of their own (more): the cases lie
at, just below and just above each limit, at a single supercell and at counts that fill no block or vector.
The second resort finds the histogram that the first one reset.
"""
from __future__ import annotations

import numpy as np
import pytest

import oracle_ref
from spearhed_amd import capi
from spearhed_amd.particles import ParticleSet
from spearhed_amd.stepper import Context


@pytest.mark.gpu
@pytest.mark.parametrize("cells", [(1, 1, 1), (7, 1, 1), (11, 31, 3), (32, 32, 1), (41, 5, 5), (45, 14, 13),
                                   (32, 16, 16), (241, 17, 2), (47, 19, 23), (128, 64, 64), (129, 64, 64)])
@pytest.mark.parametrize("n", [1, 5003])
def test_cell_starts_over_cell_counts(cells, n):
    rng = np.random.default_rng(n + cells[0])
    e = 0.125
    cfg = capi.make_config(box_len=tuple(c * e for c in cells), periodic=(0, 0, 0), kernel=capi.KERNEL_WENDLAND,
                           h0=0.499 * e, mhd=0)
    ps = ParticleSet(n)
    ps.id = rng.permutation(n).astype(np.uint64)
    ps.pos = rng.uniform(0.0, 1.0, (3, n)) * (np.array(cells)[:, None] * e)
    ps.mass[:] = 1.0 / n
    ps.h[:] = 0.499 * e
    ps.rho[:] = 1
    ps.u[:] = 1
    assert tuple(oracle_ref.grid(cfg).n[:]) == cells
    key = oracle_ref.bin_keys(cfg, "mixed", ps.pos)
    perm, cs = oracle_ref.sort_perm(key, ps.id, int(np.prod(cells)))
    print(f"cells {cells} n={n}", flush=True)
    with Context([cfg], [n], precision="mixed") as ctx:
        ctx.upload(0, ps)
        for _ in range(2):
            ctx.resort()
            k, c = ctx.sort_info(0)
            assert np.array_equal(c, cs), "cell starts differ"
            assert np.array_equal(ctx.download(0).id, ps.id[perm]), "sort permutation differs"
            assert np.array_equal(k, key[perm]), "supercell keys differ"
