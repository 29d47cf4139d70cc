"""The order of a supercell's movers and of the holes they leave, by the count of its particles: one mask word, the
most that each lane counts by itself (4 words of 64) and one more, and more than 64 words, against the oracle.

FP64: order bit-exact, every field within 1e-12 of the oracle's after 3 steps; FP32: the same set of particles and the
split form's bounds.
"""
import numpy as np
import pytest

import oracle as O
import pica_amd as P
from test_gpu_edge_cases import _check_fp32, _check_fp64, _fp32_exact, _run_pair, _say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [P.F64, P.F32])
@pytest.mark.parametrize("n", [1, 64, 65, 128, 129, 192, 255, 256, 257, 321, 449, 512, 513, 576, 4096, 4097])
def test_movers_of_one_supercell(ctx, prec, n):
    _say("mover prefix prec=%d n=%d" % (prec, n))
    rng = np.random.default_rng(n)
    # all in the supercell in the middle, most of them on their way out
    x, u = 4.0 + 4.0 * rng.random((n, 3)), rng.standard_normal((n, 3))
    if prec == P.F32:
        x, u = _fp32_exact(x, u)
    w = (1e3 * (1.0 + np.arange(n) * 2.0 ** -20)).astype(np.float32).astype(np.float64)
    sides = _run_pair(ctx, prec, (12, 12, 12), (4, 4, 4), x, u, w, 3, P.CIC, O.ESIRKEPOV, fields=9)
    _check_fp64(*sides) if prec == P.F64 else _check_fp32(*sides, (12, 12, 12))
