"""The pinned staging of a context's copies to the host grows with the copies: from two chunks of 512 KB over eight to
eight of 1 MB, and smaller copies go through the grown one. Every byte arrives."""
import numpy as np
import pytest

import pica_amd as P

pytestmark = pytest.mark.gpu

# FP32 grids of 1.05 MB (3 slots of 512 KB), 1 MB (2), 2 MB (4), 4.2 MB (8), 12 MB (8 of 1 MB), 1.6 MB (4), 6.2 MB (8), and a small one
SIZES = {"grow": [(2, 128, 1024), (2, 256, 1024), (4, 256, 1025), (3, 1000, 1024), (2, 200, 1024), (5, 310, 1000), (3, 3, 3)],
         "odd first": [(3, 29, 3011), (2, 2, 262145), (3, 1000, 1031), (2, 128, 1025)]}


@pytest.mark.parametrize("sizes", SIZES.values(), ids=SIZES.keys())
def test_staging_grows(sizes):
    ctx = P.Context(0)
    for i, size in enumerate(sizes):
        g = P.YeeGrid(ctx, size, (0.0,) * 3, (1.0,) * 3, P.F32)
        v = np.random.default_rng(i).integers(-1 << 20, 1 << 20, size).astype(np.float32)
        g.set(P.EY, v)
        for _ in range(2):
            assert np.array_equal(g.get(P.EY), v), "copy %d of %s" % (i, size)
        g.close()
    ctx.close()
