"""The last bit of the FP32 Esirkepov currents of particles that keep their node, one or two of a cell, against the same
products and sums in numpy: which products are rounded and which go unrounded into a sum is part of the result, since the
BF16 network of a denoised step turns a last bit of J into 1e-4 of its fields.

Single particles and pairs sit far apart, so that a node of J holds one rounded sum (FP64 in LDS, volume 1) exactly.
"""
import numpy as np
import pytest

import pica_amd as P

pytestmark = pytest.mark.gpu

F, L = np.float32, np.longdouble
DT = 0.5 / P.C


def _fma(a, b, c):
    """a b + c rounded once: the product is exact in 64 bits of mantissa"""
    return (np.asarray(a, F).astype(L) * np.asarray(b, F).astype(L) + np.asarray(c, F).astype(L)).astype(F)


def _shapes(shape, o, on):
    """old shape and its change on the particle's nodes, per dimension"""
    s0, s1 = (o - F(0.5)).astype(F), (on - F(0.5)).astype(F)
    if shape == P.CIC:
        f0, f1 = (np.where(s < 0, s + F(1), s).astype(F) for s in (s0, s1))
        return [F(1) - f0, f0], [(F(1) - f1) - (F(1) - f0), f1 - f0]
    half = F(0.5)
    a0, b0, a1, b1 = half - s0, half + s0, half - s1, half + s1
    S = [half * a0 * a0, _fma(-s0, s0, 0.75), half * b0 * b0]
    D = [_fma(-half * a0, a0, half * a1 * a1), _fma(-s1, s1, 0.75) - S[1], _fma(-half * b0, b0, half * b1 * b1)]
    return S, D


def _currents(shape, parts, comp, p, r):
    """running sums over the faces of component comp at the transverse nodes (p, r): parts = (o, on, q w) of each"""
    d1, d2 = (comp + 1) % 3, (comp + 2) % 3
    third, hdt, c = F(1.0) / F(3.0), F(1.0 / DT), []
    for o, on, qw in parts:
        k = (-qw) * hdt
        (S1, D1), (S2, D2) = _shapes(shape, o[:, d1], on[:, d1]), _shapes(shape, o[:, d2], on[:, d2])
        A, B = k * _fma(0.5, D1[p], S1[p]), k * _fma(third, D1[p], F(0.5) * S1[p])
        c.append(_fma(B, D2[r], A * S2[r]) if comp == 1 else _fma(A, S2[r], B * D2[r]))
    cum, out = F(0.0), []
    change = [_shapes(shape, o[:, comp], on[:, comp])[1] for o, on, _ in parts]
    for a in range(len(change[0]) - 1):
        t = change[0][a] * c[0]
        cum = cum + (_fma(change[1][a], c[1], t) if len(parts) == 2 else t)
        out.append(cum)
    return out


@pytest.mark.parametrize("ncps,spacing,edge", [(4, 8, 64), (2, 8, 64), (3, 9, 72), (8, 8, 64)])
@pytest.mark.parametrize("shape", [P.CIC, P.TSC])
@pytest.mark.parametrize("count", [1, 2])
def test_currents_to_the_last_bit(ncps, spacing, edge, shape, count):
    print("[case] split rounding ncps=%d shape=%d count=%d" % (ncps, shape, count), flush=True)
    rng = np.random.default_rng(100 * ncps + 10 * shape + count)
    at = np.stack(np.meshgrid(*[np.arange(0, edge, spacing)] * 3, indexing="ij"), -1).reshape(-1, 3)
    cell = at + rng.integers(0, min(ncps, 3), at.shape)
    # away from the node's border (TSC: the cell's, CIC: the middle), so that most stay
    lo, width = (0.55, 0.4) if shape == P.CIC else (0.1, 0.8)
    f = (lo + width * rng.random((len(cell), count, 3))).astype(F).astype(np.float64)
    x = (cell[:, None] + f).reshape(-1, 3)
    u = (0.05 * rng.standard_normal(x.shape)).astype(F).astype(np.float64)
    w = (1e8 * (1.0 + rng.random(len(x)))).astype(F).astype(np.float64)
    ctx = P.Context(0)
    ctx.set_option(P.OPT_INTERLEAVE, 0)         # slots as uploaded
    grid = P.YeeGrid.periodic(ctx, (edge,) * 3, prec=P.F32)
    ens = P.EnsembleSupercells(ctx, (edge,) * 3, (1.0,) * 3, (ncps,) * 3, prec=P.F32)
    ens.add(x, u, w)
    x0, _, w0, _ = ens.particles()
    P.particle_step(ens, grid, DT, shape, P.ESIRKEPOV)
    J = [grid.get(c) for c in (P.JX, P.JY, P.JZ)]
    x1, _, w1, _ = ens.particles()
    ctx.close()
    x1 = x1[np.argsort(w1)[np.argsort(np.argsort(w0))]]        # the slots before the step (the weights are distinct)
    x0, x1, w0 = x0.reshape(-1, count, 3), x1.reshape(-1, count, 3), w0.reshape(-1, count)

    def node(v):
        return np.floor(v - 0.5 if shape == P.CIC else v).astype(int)

    stay = np.all(node(x0) == node(x1), axis=(1, 2))
    assert stay.sum() > len(stay) // 2
    x0, x1, w0 = x0[stay], x1[stay], w0[stay]
    q = F(P.ELECTRON_CHARGE)
    parts = [((x0[:, i] - np.floor(x0[:, i])).astype(F), (x1[:, i] - np.floor(x1[:, i])).astype(F), q * w0[:, i].astype(F)) for i in range(count)]
    first = node(x0[:, 0]) + (2 if shape == P.CIC else 1)        # the lowest node's index in the array
    for comp in range(3):
        for p in range(3 if shape == P.TSC else 2):
            for r in range(3 if shape == P.TSC else 2):
                for a, want in enumerate(_currents(shape, parts, comp, p, r)):
                    i = [None] * 3
                    i[comp], i[(comp + 1) % 3], i[(comp + 2) % 3] = first[:, comp] + a + 1, first[:, (comp + 1) % 3] + p, first[:, (comp + 2) % 3] + r
                    assert np.array_equal(J[comp][tuple(i)], want), "component %d, nodes (%d, %d), face %d" % (comp, p, r, a)
