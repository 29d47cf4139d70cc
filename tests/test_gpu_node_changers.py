"""Esirkepov deposition where most particles change their node in a step, against the oracle.

A staying particle is deposited on its own nodes at once; one that changes node waits in its lane until
enough of its wavefront do.  Here momenta are relativistic in every direction, so that nearly every lane
holds a changer in every group (a lane meets its next one while the first still waits), beside a cold
plasma with a few.  Supercells of 4^3 cells (constant tile strides), other shapes, and
the largest one whose tiles fill the LDS; a last group of one particle.

FP64: order bit-exact, every field within 1e-12 of the oracle's after 3 steps (the plain path's bar).
"""
import numpy as np
import pytest

import oracle as O
import pica_amd as P
from test_gpu_edge_cases import _check_fp64, _run_pair, _say

pytestmark = pytest.mark.gpu


def _plasma(seed, ncell, n, uth):
    rng = np.random.default_rng(seed)
    x = rng.random((n, 3)) * np.asarray(ncell, np.float64)
    return x, rng.standard_normal((n, 3)) * uth, 1e4 * (1.0 + np.arange(n) * 2.0 ** -20)


@pytest.mark.parametrize("shape", [P.CIC, P.TSC])
@pytest.mark.parametrize("ncell,ncps,n,uth", [((8, 8, 8), (4, 4, 4), 4097, 2.0), ((8, 8, 8), (4, 4, 4), 700, 0.02),
                                              ((4, 8, 4), (4, 4, 4), 65, 0.3), ((6, 10, 4), (3, 5, 2), 2600, 1.0),
                                              ((12, 12, 6), (12, 12, 6), 1500, 0.5)])
def test_fp64_changers_match_oracle(ctx, shape, ncell, ncps, n, uth):
    _say("fp64 changers shape=%d ncps=%s n=%d uth=%g" % (shape, ncps, n, uth))
    x, u, w = _plasma(71 + n, ncell, n, uth)
    _check_fp64(*_run_pair(ctx, P.F64, ncell, ncps, x, u, w, 3, shape, O.ESIRKEPOV, fields=9))
