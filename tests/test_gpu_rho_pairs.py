"""Charge density where the FP32 form goes from one particle a lane to two (two to a cell on average), and where few,
some and all of a wavefront's pairs share their nodes (they are added together from 16 pairs on), against the oracle.

The bounds of the density test: 1e-13 of the largest node in FP64, 1e-7 in FP32.
"""
import numpy as np
import pytest

import oracle as O
import pica_amd as P

pytestmark = pytest.mark.gpu


def _check(ctx, prec, tol, shape, ncell, ncps, x):
    w = 1.0 + np.random.default_rng(1).integers(0, 1024, len(x)) / 1024.0
    grid = P.YeeGrid.periodic(ctx, ncell, prec=prec)
    ens = P.EnsembleSupercells(ctx, ncell, (1.0, 1.0, 1.0), ncps, prec=prec)
    ens.add(x, np.zeros_like(x), w)
    P.deposit_rho(ens, grid, shape)
    og = O.Grid.periodic(ncell)
    want = O.deposit_rho(og, O.Ensemble(ncell, ncps, (1.0, 1.0, 1.0), x, np.zeros_like(x), w), shape)
    assert np.abs(grid.get(P.RHO) - want).max() <= tol * np.abs(want).max()


@pytest.mark.parametrize("prec,tol", [(P.F64, 1e-13), (P.F32, 1e-7)])
@pytest.mark.parametrize("shape", [P.CIC, P.TSC])
@pytest.mark.parametrize("ncps,n", [((4, 4, 4), 127), ((4, 4, 4), 128), ((4, 4, 4), 129), ((3, 5, 2), 59), ((3, 5, 2), 60), ((3, 5, 2), 61)])
def test_rho_around_two_a_cell(ctx, prec, tol, shape, ncps, n):
    x = np.floor(np.random.default_rng(n).random((n, 3)) * np.asarray(ncps) * 4096.0) / 4096.0
    _check(ctx, prec, tol, shape, ncps, ncps, x)


@pytest.mark.parametrize("prec,tol", [(P.F64, 1e-13), (P.F32, 1e-7)])
@pytest.mark.parametrize("shape", [P.CIC, P.TSC])
@pytest.mark.parametrize("shared", [0, 1, 15, 16, 17, 40, 64])
def test_rho_by_pairs_that_share(ctx, prec, tol, shape, shared):
    rng = np.random.default_rng(shared)
    # 64 pairs in their slots' order (no interleave before the deposit): `shared` of them in one cell, the others in two
    a = rng.integers(0, 4, (64, 3))
    b = np.where(np.arange(64)[:, None] < shared, a, (a + [2, 0, 1]) % 4)
    x = np.stack([a, b], 1).reshape(128, 3) + rng.integers(1024, 2048, (128, 3)) / 4096.0
    x = np.concatenate([x] * 3 + [x[:1]])
    _check(ctx, prec, tol, shape, (4, 4, 4), (4, 4, 4), x)
