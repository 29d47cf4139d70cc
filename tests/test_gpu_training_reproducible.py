"""The denoiser's gradient to the last bit.

Training adds in a fixed order: the same pairs, seed and start give the same parameters, bit for bit, however the
workgroups are scheduled (a last bit that moves flips BF16 weights after some tens of iterations).

And with small whole numbers as inputs, weights and output gradients every product, sum and BF16 rounding of the
network is exact, so the device's gradient equals the oracle's exactly, in any order of adding."""
import numpy as np
import pytest

import pica_amd as P
from oracle import denoiser as D

pytestmark = pytest.mark.gpu


def _say(msg):
    print("[case] " + msg, flush=True)


def _trained(ctx, edges, batch, iters):
    rng = np.random.default_rng(3)
    low, high = (P.YeeGrid.periodic(ctx, (40, 40, 40), prec=P.F32) for _ in range(2))
    for comp in (P.JX, P.JY, P.JZ):
        f = rng.standard_normal((40, 40, 40))
        high.set(comp, np.pad(0.3 * f, 2, mode="wrap"))
        low.set(comp, np.pad(f, 2, mode="wrap"))
    dn = P.Denoiser(ctx)
    dn.init(11)
    for edge in edges:
        dn.add_pair_crops(low, high, 6, edge, edge)
    losses = dn.train(iters, batch, 1e-3, 7)
    p = dn.params()
    for h in (dn, low, high):
        h.close()
    return losses, p


# one workgroup of each layer's sums and fewer than a stride of them (9), several strides (16, 32), more bricks than
# workgroups (40, batch 8: 2400), mixed sizes (samples one by one)
@pytest.mark.parametrize("edges,batch,iters", [((9,), 1, 40), ((16,), 3, 40), ((32,), 8, 64), ((40,), 8, 24), ((12, 20), 4, 40)])
def test_training_twice_gives_the_same_bits(ctx, edges, batch, iters):
    _say("training twice edges=%s batch=%d" % (edges, batch))
    l0, p0 = _trained(ctx, edges, batch, iters)
    l1, p1 = _trained(ctx, edges, batch, iters)
    assert np.all(np.isfinite(p0)) and l0[-1] < l0[0]
    assert np.array_equal(p0.view(np.uint32), p1.view(np.uint32))
    assert np.allclose(l0, l1, rtol=2.0 ** -22, atol=0.0)      # FP64 sums of any order, rounded to FP32


def _whole_numbers(seed):
    rng = np.random.default_rng(seed)
    w = {}
    for name, shape in D.SHAPES:
        density = {"W1": 0.08, "W2": 0.01, "W3": 0.05}.get(name, 0.5)
        w[name] = rng.integers(-1, 2, shape) * (rng.random(shape) < density)
    return D.pack(w).astype(np.float32)


# one brick (4 x 4 x 16), bricks cut in every dimension, one cell, wrap-free bricks, samples that share no brick, and
# more bricks than workgroups (8 x 8 x 10)
@pytest.mark.parametrize("n,samples", [((4, 4, 16), 1), ((5, 3, 7), 1), ((4, 4, 1), 2), ((1, 1, 1), 1), ((9, 12, 48), 1),
                                       ((5, 8, 10), 3), ((8, 8, 17), 9), ((32, 32, 160), 1)])
def test_gradient_of_whole_numbers_is_exact(ctx, n, samples):
    _say("whole-number gradient n=%s samples=%d" % (n, samples))
    p = _whole_numbers(5)
    rng = np.random.default_rng(int(np.prod(n)) + samples)
    x = rng.integers(-2, 3, (samples, 3) + n).astype(np.float32)
    s = rng.integers(-1, 2, (samples, 3) + n)
    nv = int(np.prod(n))
    y, ref = np.empty_like(x), 0.0
    for k in range(samples):
        out, c = D.net_forward(p, x[k])
        # g3 = bf16(2 (out - y) / count) = s, on the device over all samples and in the oracle over one
        y[k] = out - s[k] * (1.5 * nv * samples)
        ref = ref + D.net_grad(p, x[k], out - s[k] * (1.5 * nv))[1]
        assert max(c["a1"].max(), c["a2"].max()) <= 256 and np.abs(y[k]).max() < 2 ** 22
    assert np.abs(ref).max() < 2 ** 22 and np.array_equal(ref, np.round(ref))
    dn = P.Denoiser(ctx)
    dn.set_params(p)
    got = dn.grad_batch(x, y)[1]
    dn.close()
    assert np.any(ref) and np.array_equal(got, ref.astype(np.float32))
