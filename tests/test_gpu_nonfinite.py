"""Particles whose position is not finite (either sign of not-a-number and of infinity, in one axis or in all):
they have no neighbours and are nobody's, in filtered lists and in those that are not (more than 768 candidates
or 64 particles), alone in their supercell or among others, in every schedule of the pair passes.

Neighbour counts of the others are those of the same set without them. Their sums hold the same terms in
another order, so density and derivatives agree within the parity tests' 1e-5 of the sums of the terms'
magnitudes (some 300 FP32 additions at most, 300 x 2^-24 = 1.8e-5 if every one erred alike).
"""
from __future__ import annotations

import numpy as np
import pytest

from parity import assert_scaled, gpu_stages, oracle_stages
from spearhed_amd.particles import ParticleSet
from test_gpu_cell_lists import _case

VALUES = {"nan": np.nan, "-nan": -np.nan, "inf": np.inf, "-inf": -np.inf}
TUNINGS = {"chunked": {}, "balanced": dict(pair_balance=1), "cell": dict(density_chunk=512, force_chunk=128,
                                                                        pair_balance=2)}


def _with_bad(ps, value):
    """ps and two more particles: one off in x, one in every axis."""
    out = ParticleSet(ps.n + 2)
    for name in ("id", "mask", "species", "mass", "rho", "h", "u", "psi"):
        col = getattr(ps, name)
        setattr(out, name, np.concatenate([col, col[:2]]))
    for name in ("pos", "vel", "B"):
        col = getattr(ps, name)
        setattr(out, name, np.concatenate([col, col[:, :2]], axis=1))
    out.id[-2:] = [ps.n, ps.n + 1]
    out.pos[0, -2] = value
    out.pos[:, -1] = value
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("tuning", list(TUNINGS))
@pytest.mark.parametrize("precision", ["mixed", "fp32"])
@pytest.mark.parametrize("value", list(VALUES))
@pytest.mark.parametrize("per_cell,variant", [(3, "full"), (3, "holes"), (21, "two_h"), (28, "walls"), (29, "full"),
                                              (65, "holes")])
def test_nonfinite_positions_have_no_neighbours(per_cell, variant, value, precision, tuning):
    cfg, ps = _case(per_cell, variant)
    print(f"per_cell {per_cell} {variant} {value} {precision} {tuning}", flush=True)
    bad = _with_bad(ps, VALUES[value])
    assert np.signbit(bad.pos[0, -1]) == (value[0] == "-")
    ref = gpu_stages(cfg, ps, precision, tuning=TUNINGS[tuning])
    got = gpu_stages(cfg, bad, precision, tuning=TUNINGS[tuning])
    assert not got.nnb[ps.n:].any()
    assert not got.dvdt[:, ps.n:].any() and not got.dudt[ps.n:].any()
    assert np.isfinite(got.rho[ps.n:]).all() and (got.rho[ps.n:] > 0).all()
    assert np.array_equal(got.nnb[:ps.n], ref.nnb)
    o = oracle_stages(cfg, ps, "mixed" if precision == "mixed" else "plain")
    order = o.by_id()
    for name, scale in (("rho", o.sc_rho), ("dvdt", o.sc_a), ("dudt", o.sc_du), ("dbdt", o.sc_db),
                        ("divb", o.sc_divb)):
        assert_scaled(getattr(got, name)[..., :ps.n], getattr(ref, name), scale[order] + 1e-30, name)
    assert np.all(np.abs(got.vsig[:ps.n] - ref.vsig) <= 1e-5 * ref.vsig)
