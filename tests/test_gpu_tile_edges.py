"""GPU: kernels whose tiling depends on the grid, at the sizes where a tile can go wrong."""
from __future__ import annotations

import numpy as np
import pytest

from tests._helpers import from_dev, random_state, to_dev

pytestmark = pytest.mark.gpu

OPT = (2, False, False, 0, False, False, 1)


def _case(nx, ny, nz, passive, seed=3):
    from lex_amd import _lib
    gr, phys, base = random_state(nx, ny, nz, seed=seed, passive=passive, vel=2.0)
    g = _lib.grid(nx, ny, nz, gr.dx, gr.dy, gr.dz)
    return g, tuple(to_dev(a) for a in phys), tuple(to_dev(a) for a in base[:5])


# marches of 1, 2, 5, 9 and 16 cells with full and partial last tiles, ny mod 4 of 0..3,
# one, two and three waves per column
@pytest.mark.parametrize("shape,passive", [((8, 9, 16), 0), ((40, 41, 40), 0), ((67, 62, 64), 2), ((97, 91, 70), 1),
                                           ((157, 160, 130), 2)], ids=str)
def test_stage_tiles_equal_per_operator_kernels(shape, passive):
    """One step with the stage kernel against one kernel per reference routine: the same
    arithmetic up to operation order, a few FP32 ulps of each field (64, as for the other
    fused kernels)."""
    from lex_amd import one_sprint_functions as sp
    g, phys, base = _case(*shape, passive)
    got = sp.fused_step(tuple(a.clone() for a in phys), base, g, OPT, dt=0.2, n_sound=4)
    ref = sp.fused_step(tuple(a.clone() for a in phys), base, g, OPT, dt=0.2, n_sound=4, impl=1)
    for q, (a, b) in enumerate(zip(got, ref)):
        a, b = from_dev(a), from_dev(b)
        assert np.isfinite(b).all()
        ulp = float(np.spacing(np.float32(np.abs(b).max())))
        assert np.max(np.abs(a - b)) <= 64 * ulp, (q, np.max(np.abs(a - b)) / ulp)
