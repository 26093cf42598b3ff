"""The kick on both sides of the number of workgroups up to which it finalises its runs itself (64 of 256
particles), against the same run batched with a large one, whose runs a launch of their own finalises: state,
times and conserved sums are equal bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_kick_finalize import _result, _run


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["mixed", "fp32"])
@pytest.mark.parametrize("n", [63 * 256, 64 * 256 - 1, 64 * 256, 64 * 256 + 1])
def test_kick_on_both_sides_of_the_limit(n, precision):
    print(f"n {n} {precision}", flush=True)
    own = _run(n)
    a, sums_a, end_a = _result([own], precision)
    b, sums_b, end_b = _result([own, _run(65600)], precision)
    for name in ("id", "pos", "vel", "u", "rho", "B", "psi", "dvdt", "vsig"):
        assert np.array_equal(getattr(a, name), getattr(b, name)), name
    assert sums_a == sums_b and end_a == end_b
