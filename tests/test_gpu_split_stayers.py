"""FP32 Esirkepov deposition of staying particles, alone and in pairs, against the FP64 oracle.

Sizes where the tiles or the pairing could go wrong: 4^3 supercells (component-interleaved tile rows) and
other shapes (plain rows), cells with one, two and an odd number of particles (lanes whose second particle is
missing or sits in another cell), and a hot dense plasma whose node changers overflow the change queue.
The bounds are the split form's per-quantity bounds.
"""
import pytest

import oracle as O
import pica_amd as P
from test_gpu_split import _compare, _say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [P.CIC, P.TSC])
@pytest.mark.parametrize("ncell,ncps,ppc,uth", [((8, 8, 8), (4, 4, 4), 1, 0.01), ((8, 4, 12), (4, 4, 4), 5, 0.01),
                                                ((8, 8, 4), (4, 4, 4), 40, 0.5), ((8, 8, 8), (2, 2, 2), 3, 0.05),
                                                ((8, 8, 16), (8, 8, 8), 2, 0.05), ((10, 9, 4), (5, 3, 4), 7, 0.05)])
def test_stayers_match_oracle(ctx, shape, ncell, ncps, ppc, uth):
    _say("stayers shape=%d ncps=%s ppc=%d uth=%g" % (shape, ncps, ppc, uth))
    _compare(ctx, shape, O.ESIRKEPOV, ncell, ncps, ppc, 4, 311 + ppc, uth=uth)


@pytest.mark.parametrize("dep", [P.DIRECT, P.ESIRKEPOV])
def test_direct_and_esirkepov_tiles(ctx, dep):
    _compare(ctx, P.TSC, dep, (8, 12, 4), (4, 4, 4), 3, 4, 77, uth=0.02)
