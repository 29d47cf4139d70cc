"""Particle steps of two-dimensional runs whose tiles take other strides than the conflict-free ones, since those
would cost a workgroup on the CU: long, wide and large supercells of one cell in z, against the oracle, with few
particles and with so many that the mover mask adds to the LDS.

FP64: order bit-exact, every field within 1e-12 of the oracle's after 3 steps; FP32: the split form's bounds.
"""
import numpy as np
import pytest

import oracle as O
import pica_amd as P
from test_gpu_edge_cases import _check_fp64, _run_pair, _say
from test_gpu_split import _compare

pytestmark = pytest.mark.gpu

SHAPES = [((24, 4, 1), (12, 2, 1)), ((12, 8, 1), (12, 4, 1)), ((8, 12, 1), (4, 12, 1)), ((9, 18, 1), (9, 9, 1)), ((12, 5, 1), (6, 5, 1))]


@pytest.mark.parametrize("ncell,ncps", SHAPES)
@pytest.mark.parametrize("shape", [P.CIC, P.TSC])
@pytest.mark.parametrize("dep", [O.DIRECT, O.ESIRKEPOV])
def test_fp64_levels_match_oracle(ctx, ncell, ncps, shape, dep):
    _say("flat levels fp64 ncps=%s shape=%d dep=%d" % (ncps, shape, dep))
    for n in (300, 6000):
        rng = np.random.default_rng(n)
        x, w = rng.random((n, 3)) * np.asarray(ncell, np.float64), 1e3 * (1.0 + np.arange(n) * 2.0 ** -20)
        _check_fp64(*_run_pair(ctx, P.F64, ncell, ncps, x, rng.standard_normal((n, 3)) * 0.1, w, 3, shape, dep, fields=9))


@pytest.mark.parametrize("ncell,ncps", SHAPES)
@pytest.mark.parametrize("shape", [P.CIC, P.TSC])
@pytest.mark.parametrize("dep", [O.DIRECT, O.ESIRKEPOV])
def test_fp32_levels_match_oracle(ctx, ncell, ncps, shape, dep):
    _compare(ctx, shape, dep, ncell, ncps, 6, 4, 43, uth=0.02)
