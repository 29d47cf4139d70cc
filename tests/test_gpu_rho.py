"""Charge density against the oracle: pairs of particles that share their nodes and pairs that do not, a last slot
without a partner, supercells with constant and with run-time tile strides, empty supercells.

The sums are FP64 in both: the nodes agree within 1e-13 of the largest (some hundred terms of 2^-53 each) in FP64;
the FP32 grid rounds the same sum once (2^-24), and the FP32 form's offsets are exact here (multiples of 2^-12).
"""
import numpy as np
import pytest

import oracle as O
import pica_amd as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec,tol", [(P.F64, 1e-13), (P.F32, 1e-7)])
@pytest.mark.parametrize("shape", [P.CIC, P.TSC])
@pytest.mark.parametrize("ncell,ncps,n", [((8, 8, 4), (4, 4, 4), 1), ((8, 4, 12), (4, 4, 4), 513), ((4, 8, 4), (4, 4, 4), 4001),
                                          ((6, 5, 8), (3, 5, 2), 777), ((12, 12, 1), (6, 6, 1), 1300)])
def test_rho_matches_oracle(ctx, prec, tol, shape, ncell, ncps, n):
    rng = np.random.default_rng(n)
    x = np.floor(rng.random((n, 3)) * np.asarray(ncell) * 4096.0) / 4096.0
    x[n // 3:] = x[np.arange(n // 3, n) % max(n // 3, 1)] // 1 + rng.integers(0, 4096, (n - n // 3, 3)) / 4096.0   # shared cells
    u, w = np.zeros((n, 3)), 1.0 + rng.integers(0, 1024, n) / 1024.0
    grid = P.YeeGrid.periodic(ctx, ncell, prec=prec)
    ens = P.EnsembleSupercells(ctx, ncell, (1.0, 1.0, 1.0), ncps, prec=prec)
    ens.add(x, u, w)
    P.deposit_rho(ens, grid, shape)
    got = grid.get(P.RHO)
    og = O.Grid.periodic(ncell)
    want = O.deposit_rho(og, O.Ensemble(ncell, ncps, (1.0, 1.0, 1.0), x, u, w), shape)
    assert np.abs(got - want).max() <= tol * np.abs(want).max()
