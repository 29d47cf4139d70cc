"""A batch whose ensembles changed between two runs, against stepping each pair on its own: supercells of one of them
re-bucketed, so that the batch holds several shapes at once; and, with nothing else that would prepare the launches
again, particles uploaded, loaded from a snapshot, re-bucketed or stepped on their own, or other species.

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


def _upload(ctx, pair, tmp_path, dt):
    rng = np.random.default_rng(5)
    e, _ = pair
    n = 4000          # more than before: other buffers, other capacities
    e.add(rng.random((n, 3)) * e.ncell, 0.05 * rng.standard_normal((n, 3)), 1e3 * (1.0 + np.arange(n) * 2.0 ** -20))


def _reload(ctx, pair, tmp_path, dt):
    pair[0].save(str(tmp_path / "e"))
    pair[0].load(str(tmp_path / "e"))


def _rebucket(ctx, pair, tmp_path, dt):
    pair[0].set_supercells((2, 4, 2))


def _own_steps(ctx, pair, tmp_path, dt):
    pair[0].set_slack(0.0, 0)
    pair[0].set_supercells((2, 2, 2))
    P.run(pair[0], pair[1], dt, 3, P.TSC, P.ESIRKEPOV)         # overflows its supercells: rebuilt


def _other_species(ctx, pair, tmp_path, dt):
    ctx.set_species([3.0 * P.ELECTRON_MASS], [2.0 * P.ELECTRON_CHARGE])


@pytest.mark.parametrize("prec", [P.F64, P.F32])
@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("change", [_upload, _reload, _rebucket, _own_steps, _other_species])
def test_changed_between_runs_of_one_dt(prec, graph, change, tmp_path):
    _say("batch, %s between two runs, prec=%d graph=%d" % (change.__name__, prec, graph))
    dt = courant_dt()
    ctx = P.Context(0)
    ctx.set_option(P.OPT_INTERLEAVE, 0)
    if change is _other_species:
        ctx.set_species([P.ELECTRON_MASS], [P.ELECTRON_CHARGE])
    mine, ref = _pairs(ctx, prec), _pairs(ctx, prec)
    b = P.Batch(ctx, mine)
    b.set(P.BATCH_GRAPH, graph)
    b.run(dt, 2, P.TSC, P.ESIRKEPOV)
    for e, g in ref:
        P.run(e, g, dt, 2, P.TSC, P.ESIRKEPOV)
    for pair in (mine[1], ref[1]):
        change(ctx, pair, tmp_path, dt)
    b.run(dt, 3, P.TSC, P.ESIRKEPOV)
    for e, g in ref:
        P.run(e, g, dt, 3, P.TSC, P.ESIRKEPOV)
    _same(prec, mine, ref, change.__name__)
    ctx.close()
