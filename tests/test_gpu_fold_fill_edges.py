"""The periodic step's one-launch fold and fill of J, and the Yee updates' ghost images, on grids whose edges are
around the ghost width, against the oracle: one to five cells (a cell there has up to four ghosts along a
dimension), mixed with longer ones, in the single and the batched step.

FP64: every field with its ghosts within 1e-12 of the oracle's after 3 steps (the plain path's bar).
"""
import numpy as np
import pytest

import oracle as O
import pica_amd as P
from test_gpu_edge_cases import _check_fp64, _run_pair, _say

pytestmark = pytest.mark.gpu

GRIDS = [(1, 1, 6), (1, 5, 1), (6, 1, 7), (2, 3, 4), (3, 3, 3), (5, 4, 2), (8, 1, 1), (4, 4, 4), (5, 9, 6)]


def _plasma(ncell):
    rng = np.random.default_rng(int(np.dot(ncell, (1, 10, 100))))
    n = 6 * int(np.prod(ncell)) + 1
    return rng.random((n, 3)) * np.asarray(ncell, np.float64), rng.standard_normal((n, 3)) * 0.2, 1e4 * (1.0 + np.arange(n) * 2.0 ** -20)


@pytest.mark.parametrize("ncell", GRIDS)
@pytest.mark.parametrize("shape,dep", [(P.CIC, O.DIRECT), (P.TSC, O.ESIRKEPOV)])
def test_small_edges_match_oracle(ctx, ncell, shape, dep):
    _say("fold fill ncell=%s shape=%d dep=%d" % (ncell, shape, dep))
    x, u, w = _plasma(ncell)
    _check_fp64(*_run_pair(ctx, P.F64, ncell, ncell, x, u, w, 3, shape, dep, fields=9))


@pytest.mark.parametrize("prec", [P.F64, P.F32])
def test_batch_ghosts_equal_the_cells_they_image(ctx, prec):
    n = (4, 8, 4)
    x, u, w = _plasma(n)
    grid = P.YeeGrid.periodic(ctx, n, prec=prec)
    ens = P.EnsembleSupercells(ctx, n, (1.0, 1.0, 1.0), (4, 4, 4), prec=prec)
    ens.add(x, u, w)
    P.Batch(ctx, [(ens, grid)]).run(0.5 / P.C, 3, P.TSC, P.ESIRKEPOV)
    for comp in range(9):
        f = grid.get(comp)
        assert np.abs(f).max() > 0.0
        assert np.array_equal(f, np.pad(f[2:-2, 2:-2, 2:-2], 2, mode="wrap")), "component %d" % comp
