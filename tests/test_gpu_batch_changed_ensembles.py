"""A batch whose ensembles changed between two runs, against stepping each pair on its own: supercells of one of them
re-bucketed, so that the batch holds several shapes at once.

Same bounds as the batch tests: FP64 1e-12, FP32 2e-5 of the scale, supercell membership and particle order equal."""
import numpy as np
import pytest

import pica_amd as P
from helpers import courant_dt
from test_gpu_batch import _compare, _no_interleave, _pairs, _say, _state      # noqa: F401 (autouse fixture)

pytestmark = pytest.mark.gpu

FORMS = [(P.TSC, P.ESIRKEPOV), (P.CIC, P.DIRECT)]


def _same(prec, mine, ref, what):
    for i, ((e, g), (re_, rg)) in enumerate(zip(mine, ref)):
        _compare(prec, _state(e, g), _state(re_, rg), "%s, ensemble %d" % (what, i))


# the first ensemble keeps 4^3 supercells and another leaves them, the first leaves them, all but one do
@pytest.mark.parametrize("prec", [P.F64, P.F32])
@pytest.mark.parametrize("shape,dep", FORMS)
@pytest.mark.parametrize("change", [{1: (2, 2, 2)}, {2: (8, 4, 8)}, {0: (2, 2, 2)}, {0: (8, 8, 12), 1: (2, 4, 8), 3: (4, 8, 4)}])
def test_supercells_of_one_ensemble_change(ctx, prec, shape, dep, change):
    _say("batch of mixed supercells prec=%d shape=%d dep=%d %s" % (prec, shape, dep, change))
    dt = courant_dt()
    mine, ref = _pairs(ctx, prec), _pairs(ctx, prec)
    b = P.Batch(ctx, mine)
    b.run(dt, 2, shape, dep)
    for e, g in ref:
        P.run(e, g, dt, 2, shape, dep)
    for i, ncps in change.items():
        mine[i][0].set_supercells(ncps)
        ref[i][0].set_supercells(ncps)
    b.run(0.5 * dt, 3, shape, dep)          # another dt: the launches are prepared again
    for e, g in ref:
        P.run(e, g, 0.5 * dt, 3, shape, dep)
    _same(prec, mine, ref, "re-bucketed")
    b.close()
