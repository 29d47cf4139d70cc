"""Copies to ordinary host memory go through pinned chunks: every byte arrives, at sizes around the
first staged one (1 MB), the chunk (512 KB, 1 MB above 6 MB), around the eight slots and of odd
length; growing the staging, several threads on one context, and a destination that is pinned already."""
import ctypes
import threading

import numpy as np
import pytest

import pica_amd as P

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (3, 3, 3), (3, 5, 7), (2, 128, 1023), (2, 128, 1024), (2, 128, 1025), (3, 3, 29137), (3, 173, 1009),
          (2, 768, 1023), (2, 768, 1024), (2, 768, 1025), (3, 1024, 768), (5, 1021, 1031)]


@pytest.fixture(scope="module")
def ctx():
    return P.Context(0)


def _grid(ctx, shape, prec):
    return P.YeeGrid(ctx, shape, (0.0,) * 3, (1.0,) * 3, prec)


def _values(shape, dtype, seed):
    r = np.random.default_rng(seed)
    return r.integers(-1 << 20, 1 << 20, shape).astype(dtype)


@pytest.mark.parametrize("prec", [P.F32, P.F64])
@pytest.mark.parametrize("shape", SHAPES)
def test_round_trip(ctx, shape, prec):
    g = _grid(ctx, shape, prec)
    for comp in (P.EX, P.BY):
        v = _values(shape, g.dtype, comp)
        g.set(comp, v)
        assert np.array_equal(g.get(comp), v)
    g.close()


def test_new_context_grows_its_staging():
    c = P.Context(0)
    for i, shape in enumerate([(2, 2, 3), (3, 1000, 1024), (2, 5, 10), (2, 100, 1024), (3, 1000, 1031)]):
        g = _grid(c, shape, P.F32)
        v = _values(shape, np.float32, i)
        g.set(P.EZ, v)
        assert np.array_equal(g.get(P.EZ), v)
        g.close()
    c.close()


def test_threads_share_a_context(ctx):
    grids = [_grid(ctx, shape, P.F32) for shape in ((2, 50, 1024), (3, 853, 1001), (3, 239, 1000))]
    vals = [_values(g.size, np.float32, i) for i, g in enumerate(grids)]
    for g, v in zip(grids, vals):
        g.set(P.EX, v)
    ctx.sync()
    bad = []

    def work(i):
        for _ in range(5):
            if not np.array_equal(grids[i].get(P.EX), vals[i]):
                bad.append(i)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad


def test_pinned_destination(ctx):
    hip = ctypes.CDLL("libamdhip64.so")
    g = _grid(ctx, (3, 101, 1013), P.F32)
    v = _values(g.size, np.float32, 9)
    g.set(P.BX, v)
    out = ctypes.c_void_p()
    assert hip.hipHostMalloc(ctypes.byref(out), ctypes.c_size_t(v.nbytes), ctypes.c_uint(0)) == 0
    ctx.check(P.lib().pk_grid_copy(g.h, P.BX, out, P.D2H))
    assert np.array_equal(np.ctypeslib.as_array(ctypes.cast(out, ctypes.POINTER(ctypes.c_float)), g.size), v)
    assert hip.hipHostFree(out) == 0
    g.close()
