"""Weight and bias gradients of the warm-start network at shapes whose chunks of
8x8-position tiles take every form of the two kernels:

  (3, 208, 176)  level 0: 429 tiles in chunks of two, so a workgroup goes through
                 several tiles, the last used chunk has one, and 41 chunks are
                 empty; up to 429 chunks (summed by 16 threads an output), 32 and 8
                 (one thread) at the coarse levels; partial tiles
  (4, 256, 128)  512 whole tiles, chunks of two without a remainder
  (1, 48, 80)    partial tiles at every level, single-tile chunks

The network is one whose values are exact in BF16: a 3x3 layer's output channel
takes one input channel at one tap times +-1, a 1x1 layer's the difference of two
(the last layer's four channels, its output is not rounded), images and targets
are -1, 0 and 1.  An activation is then a multiple of 1/64 (three 2x2 averages),
and below 256/64 in these cases, eight bits; the oracle with and without rounding
must agree exactly.  Rounding thus moves neither side, and the GPU's sums over
positions differ from the CPU oracle's by FP32 additions alone: at most 600 of
them one after another (128 positions of a chunk, 429 chunks), each within 2^-24
of the sum of the absolute terms.  That is the bar, element by element; a tile left
out or added twice moves an element by about 1/512 of that sum.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def exact_network(wo, rng):
    p = []
    for li, (ks, cin, cout, _, _) in enumerate(wo.LAYERS):
        w = np.zeros((ks * ks, cout, cin), np.float32)
        used = 8 if li == 10 else cout  # the last layer's other outputs stay zero
        co, shift = np.arange(used), rng.integers(cin)
        for k in range(4 if li == 10 else (1 if ks == 3 else 2)):  # every input channel is taken
            sign = rng.choice([-1.0, 1.0, 1.0], used) if ks == 3 else (-1.0) ** k
            w[rng.integers(ks * ks, size=used), co, (co * 5 + k * used + shift) % cin] = sign
        p += [w.ravel(), np.zeros(cout, np.float32)]
    return np.concatenate(p)


@pytest.mark.parametrize("shape", [(3, 208, 176), (4, 256, 128), (1, 48, 80)])
def test_gradients_match_oracle_term_by_term(shape, monkeypatch):
    import isg
    from oracle import warmnet_oracle as wo
    print("warm-start network gradients", shape, flush=True)
    rng = np.random.default_rng(21)
    x = rng.integers(-1, 2, shape + (8,)).astype(np.float32)
    t = rng.integers(-1, 2, shape + (2,)).astype(np.float32)
    n = isg.WarmNet(max_batch=shape[0], max_pixels=shape[1] * shape[2])
    n.scales = np.ones(9, np.float32)
    n.params = exact_network(wo, rng)
    loss = n.loss_grad(x, t)
    g = n.grads()
    sums, plain = [], wo.wgrad

    def wgrad(dpre, inp, ks, rnd):  # called from the last layer to the first
        gw, gb = plain(np.abs(dpre), np.abs(inp), ks, rnd)
        sums.insert(0, np.concatenate([gw.ravel(), gb]))
        return plain(dpre, inp, ks, rnd)

    monkeypatch.setattr(wo, "wgrad", wgrad)
    ones = np.ones(9, np.float32)
    np.testing.assert_array_equal(wo.forward(n.params, x, ones, rnd=True)["y"], wo.forward(n.params, x, ones, rnd=False)["y"])
    lref, gref = wo.loss_grad(n.params, x, t, ones, rnd=True)
    assert lref > 0 and abs(loss - lref) < 1e-6 * lref  # differences exact, their squares summed in float64
    bar = 600 * 2.0 ** -24 * np.concatenate(sums)
    for li, (w, b) in enumerate(wo.offsets()[0]):
        for name, a, e in (("weights", w, b), ("bias", b, b + wo.LAYERS[li][2])):
            d = np.abs(g[a:e] - gref[a:e])
            print("layer %d %s: %d of %d nonzero, largest error %.2e of its bar" %
                  (li, name, np.count_nonzero(gref[a:e]), e - a, np.max(d / np.maximum(bar[a:e], 1e-300))), flush=True)
            assert np.count_nonzero(gref[a:e]) > 0 and (d <= bar[a:e]).all()
