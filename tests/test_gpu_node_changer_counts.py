"""FP64 Esirkepov deposition with a given number of node changers in each wavefront's group of 64, against the oracle:
none, fewer than the four that are deposited together, around the count from which every changer is deposited by its
own lane (8 with CIC, 16 with TSC), and all.

Order bit-exact, every field within 1e-12 of the oracle's after 2 steps (the plain path's bar).
"""
import numpy as np
import pytest

import oracle as O
import pica_amd as P
from helpers import courant_dt
from test_gpu_edge_cases import _check_fp64, _run_pair, _say

pytestmark = pytest.mark.gpu

COUNTS = (0, 1, 3, 4, 5, 7, 8, 9, 12, 15, 16, 17, 31, 63, 64)


def _groups(shape, counts, seed):
    """64 particles a group, in one supercell; `count` of a group's cross their node's border along x, y or z"""
    rng = np.random.default_rng(seed)
    x, u = [], []
    stay, cross = (0.1, 0.3) if shape == P.CIC else (0.5, 0.9)
    for k in counts:
        mover = np.zeros(64, bool)
        mover[rng.permutation(64)[:k]] = True
        f = np.where(mover[:, None], cross, stay) + rng.uniform(-0.05, 0.05, (64, 3))
        x.append(rng.integers(0, 4, (64, 3)) + f)
        v = 0.01 * rng.standard_normal((64, 3))
        v[mover, rng.integers(0, 3, k)] += 2.0
        u.append(v)
    x, u = np.concatenate(x), np.concatenate(u)
    moved = x + u / np.sqrt(1.0 + (u * u).sum(1, keepdims=True)) * P.C * courant_dt()
    node = np.floor(x - 0.5) if shape == P.CIC else np.floor(x)
    change = np.any((np.floor(moved - 0.5) if shape == P.CIC else np.floor(moved)) != node, 1)
    assert np.array_equal(change.reshape(-1, 64).sum(1), counts)
    return x, u, 1e2 * (1.0 + np.arange(len(x)) * 2.0 ** -20)


@pytest.mark.parametrize("shape", [P.CIC, P.TSC])
@pytest.mark.parametrize("ncps", [(4, 4, 4), (4, 4, 2)])
def test_counts_of_changers(ctx, shape, ncps):
    _say("node changers by count shape=%d ncps=%s" % (shape, ncps))
    for counts in [(k,) for k in COUNTS] + [COUNTS]:
        x, u, w = _groups(shape, counts, 5 + sum(counts))
        _check_fp64(*_run_pair(ctx, P.F64, (4, 4, 4), ncps, x, u, w, 2, shape, O.ESIRKEPOV, fields=9))
