"""The batched step on grids whose edges are around the ghost width (one to four cells, mixed with longer ones) and on
two-dimensional ones, against the oracle: every component with its ghosts.

FP64: order bit-exact, every field within 1e-12 of the oracle's after 3 steps (the plain path's bar); FP32: within
2e-5 of the single step's (the batch tests' bar), ghosts equal to the cells that they image.
"""
import numpy as np
import pytest

import oracle as O
import pica_amd as P
from helpers import courant_dt, random_fields, rel_err
from test_gpu_edge_cases import _check_fp64, _say

pytestmark = pytest.mark.gpu

GRIDS = [((2, 3, 4), (2, 3, 4)), ((8, 1, 1), (4, 1, 1)), ((1, 1, 6), (1, 1, 3)), ((1, 5, 1), (1, 5, 1)), ((6, 1, 7), (3, 1, 7)), ((3, 3, 3), (3, 3, 3)),
         ((12, 12, 1), (6, 6, 1)), ((24, 4, 1), (12, 2, 1))]


def _input(ncell, n=400):
    rng = np.random.default_rng(int(np.dot(ncell, (1, 10, 100))))
    return rng.random((n, 3)) * np.asarray(ncell, np.float64), rng.standard_normal((n, 3)) * 0.2, 1e4 * (1.0 + np.arange(n) * 2.0 ** -20)


@pytest.mark.parametrize("ncell,ncps", GRIDS)
@pytest.mark.parametrize("shape,dep", [(P.CIC, O.DIRECT), (P.TSC, O.ESIRKEPOV)])
def test_batch_matches_oracle(ctx, ncell, ncps, shape, dep):
    _say("batch small edges ncell=%s shape=%d dep=%d" % (ncell, shape, dep))
    dt, (x, u, w) = courant_dt(), _input(ncell)
    og = O.Grid.periodic(ncell)
    random_fields(np.random.default_rng(9), og, 3e-3, 3e-3)
    oe = O.Ensemble(ncell, ncps, (1.0, 1.0, 1.0), x, u, w)
    pairs = []
    for _ in range(2):
        g = P.YeeGrid.periodic(ctx, ncell)
        g.set_all(og.f)
        e = P.EnsembleSupercells(ctx, ncell, (1.0, 1.0, 1.0), ncps)
        e.add(x, u, w)
        pairs.append((e, g))
    P.Batch(ctx, pairs).run(dt, 3, shape, dep)
    for _ in range(3):
        O.step(og, oe, dt, shape, dep)
    for e, g in pairs:
        _check_fp64(og, oe, g, e)


@pytest.mark.parametrize("ncell,ncps", GRIDS)
def test_fp32_batch_matches_single(ctx, ncell, ncps):
    _say("batch small edges fp32 ncell=%s" % (ncell,))
    sides = []
    for batch in (False, True):
        g = P.YeeGrid.periodic(ctx, ncell, prec=P.F32)
        e = P.EnsembleSupercells(ctx, ncell, (1.0, 1.0, 1.0), ncps, prec=P.F32)
        e.add(*_input(ncell))
        if batch:
            P.Batch(ctx, [(e, g)]).run(courant_dt(), 3, P.TSC, P.ESIRKEPOV)
        else:
            P.run(e, g, courant_dt(), 3, P.TSC, P.ESIRKEPOV)
        sides.append(g.get_all())
    for c in range(9):
        f = sides[1][c]
        assert np.array_equal(f, np.pad(f[2:-2, 2:-2, 2:-2], 2, mode="wrap")), "component %d" % c
    for comps in ((0, 1, 2), (3, 4, 5), (6, 7, 8)):
        scale = max(np.abs(sides[0][c]).max() for c in comps)
        assert max(np.abs(sides[1][c] - sides[0][c]).max() for c in comps) <= 2e-5 * scale
