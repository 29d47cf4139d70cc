"""Particle steps of two-dimensional runs (supercells of one cell in z), whose tiles have strides of their own,
against the oracle: square and oblong supercells, one row or one cell, and the largest.

FP64: order bit-exact, every field within 1e-12 of the oracle's after 3 steps; FP32: the split form's bounds.
"""
import numpy as np
import pytest

import oracle as O
import pica_amd as P
from test_gpu_edge_cases import _check_fp64, _run_pair, _say
from test_gpu_split import _compare

pytestmark = pytest.mark.gpu

SHAPES = [((12, 12, 1), (6, 6, 1), 1700), ((10, 9, 1), (5, 3, 1), 400), ((8, 4, 1), (1, 4, 1), 130), ((4, 6, 1), (4, 1, 1), 129),
          ((3, 3, 1), (1, 1, 1), 50), ((24, 12, 1), (12, 12, 1), 900), ((14, 21, 1), (2, 7, 1), 700)]


@pytest.mark.parametrize("ncell,ncps,n", SHAPES)
@pytest.mark.parametrize("shape", [P.CIC, P.TSC])
@pytest.mark.parametrize("dep", [O.DIRECT, O.ESIRKEPOV])
def test_fp64_flat_matches_oracle(ctx, ncell, ncps, n, shape, dep):
    _say("flat ncps=%s shape=%d dep=%d" % (ncps, shape, dep))
    rng = np.random.default_rng(n)
    x, w = rng.random((n, 3)) * np.asarray(ncell, np.float64), 1e4 * (1.0 + np.arange(n) * 2.0 ** -20)
    _check_fp64(*_run_pair(ctx, P.F64, ncell, ncps, x, rng.standard_normal((n, 3)) * 0.1, w, 3, shape, dep, fields=9))


@pytest.mark.parametrize("ncell,ncps", [((12, 12, 1), (6, 6, 1)), ((10, 9, 1), (5, 3, 1)), ((8, 4, 1), (1, 4, 1)), ((12, 12, 1), (12, 12, 1))])
@pytest.mark.parametrize("shape", [P.CIC, P.TSC])
@pytest.mark.parametrize("dep", [O.DIRECT, O.ESIRKEPOV])
def test_fp32_flat_matches_oracle(ctx, ncell, ncps, shape, dep):
    _compare(ctx, shape, dep, ncell, ncps, 6, 4, 41, uth=0.02)
