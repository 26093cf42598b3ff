"""Two particles as close as FP32 separations go, approaching each other: signal speed and derivatives against the
oracle while r^2 is a normal number, and the signal speed c_i + c_j + beta |dv| in closed form; below that r^2 has
lost its digits and the results are finite."""
from __future__ import annotations

import numpy as np
import pytest

from parity import compare_forces, gpu_stages, oracle_stages
from spearhed_amd import capi
from spearhed_amd.particles import ParticleSet

KERNELS = {"cubic": capi.KERNEL_CUBIC, "quintic": capi.KERNEL_QUINTIC, "wendland": capi.KERNEL_WENDLAND}


def _pair(d, kernel, two_h):
    ps = ParticleSet(2)
    ps.pos[0] = [0.0, d]
    ps.mass[:] = 1.0
    ps.h[:] = [0.1, 0.09 if two_h else 0.1]
    ps.u[:] = 1.0
    ps.rho[:] = 1.0
    ps.vel[0] = [0.5, -0.5]
    cfg = capi.make_config(box_len=(2, 2, 2), periodic=(0, 0, 0), kernel=KERNELS[kernel], h0=0.1, mhd=0)
    return cfg, ps


@pytest.mark.gpu
@pytest.mark.parametrize("two_h", [False, True])
@pytest.mark.parametrize("kernel", list(KERNELS))
@pytest.mark.parametrize("prec", ["mixed", "plain"])
@pytest.mark.parametrize("d", [1e-15, 4e-19, 3e-19, 2e-19, 1.2e-19, 1.09e-19])
def test_close_pair_against_the_oracle(d, prec, kernel, two_h):
    cfg, ps = _pair(d, kernel, two_h)
    print(f"d {d} {prec} {kernel} two_h {two_h}", flush=True)
    g = gpu_stages(cfg, ps, "fp32" if prec == "plain" else prec)
    c = np.sqrt(cfg.gamma * (cfg.gamma - 1.0) * ps.u.astype(np.float64))
    assert np.all(np.abs(g.vsig - (c.sum() + cfg.beta_visc * 1.0)) <= 1e-5 * g.vsig)
    compare_forces(g, oracle_stages(cfg, ps, prec), mhd=False)


@pytest.mark.gpu
@pytest.mark.parametrize("kernel", list(KERNELS))
@pytest.mark.parametrize("d", [1e-19, 1e-20, 1e-22, 1e-30, 0.0])
def test_closer_pairs_are_finite(d, kernel):
    cfg, ps = _pair(d, kernel, False)
    print(f"d {d} {kernel}", flush=True)
    g = gpu_stages(cfg, ps, "mixed")
    for name in ("rho", "dvdt", "dudt", "vsig"):
        assert np.isfinite(getattr(g, name)).all(), name
    assert g.nnb.tolist() == [1, 1]
