"""The network's gradient where every sum is exact: small whole numbers for
parameters, inputs and the differences from the target, a power of two of
pixels in the loss.  All products are then whole multiples of one power of two
whose sums stay below 2^24 of it (checked), so FP32 adds them without rounding
in any order, what is rounded to BF16 is the same number on both sides, and the
kernels have to give the reference's gradient bit for bit."""
import numpy as np
import pytest

import cnn_ref as R
import pvof

pytestmark = pytest.mark.gpu


def whole_params(seed):
    rng = np.random.default_rng(seed)
    p = np.zeros(R.NPARAM)

    def put(a, b, density):
        p[a:b] = rng.integers(-1, 2, b - a) * (rng.random(b - a) < density)

    put(0, 864, 0.3)
    put(864, 896, 1.0)
    for k in range(4):
        o = 896 + k * 9248
        put(o, o + 9216, 0.03)
        put(o + 9216, o + 9248, 1.0)
    put(37888, 38176, 0.2)
    put(38176, 38177, 1.0)
    return p


# one tile; a row of tiles; the most rows of partials (1024) exactly; half of
# the workgroups with two tiles (1536 tiles: 8 images of 6, 32 times over)
@pytest.mark.parametrize("images,copies,h,w,border", [(1, 1, 16, 16, 4), (1, 1, 16, 16, 0), (2, 1, 16, 64, 0),
                                                      (8, 128, 16, 16, 4), (8, 32, 32, 48, 8)])
@pytest.mark.parametrize("px", [0, 1])
def test_gradient_is_exact(gpu, images, copies, h, w, border, px):
    rng = np.random.default_rng(images * copies * h * w + px)
    p = whole_params(images + 10 * copies + px)
    x = rng.integers(-2, 3, (images, h, w, 3)).astype(np.float64)
    out, acts = R.forward(p, x, px, use_bf16=True)
    off = rng.integers(-1, 2, out.shape) * (rng.random(out.shape) < 0.25)
    tgt = out + off
    inner = (slice(None), slice(border, h - border), slice(border, w - border))
    n = out[inner].size * copies
    assert n & (n - 1) == 0
    gout = np.zeros_like(out)
    gout[inner] = -2.0 * off[inner] / n
    ref = copies * R.backward(p, acts, gout, px, use_bf16=True)
    # the largest any sum of a gradient can get, in units of 2 / n: all its terms of one sign
    big = copies * R.backward(np.abs(p), acts, np.abs(gout), px, use_bf16=True) * n / 2
    assert np.abs(out).max() < 2 ** 24 and np.abs(big).max() < 2 ** 24
    net = pvof.Network(pvof.Solver(pvof.config1_params(NXM=32, NYM=64)), seed=7)
    net.set_params(p.astype(np.float32))
    got, loss, grad = net.eval(np.concatenate([x] * copies).astype(np.float32),
                               np.concatenate([tgt] * copies).astype(np.float32), px=px, border=border, want_grad=True)
    assert np.array_equal(got, np.concatenate([out] * copies))
    assert loss == copies * (off[inner] ** 2).sum() / n
    for a, b in [(0, 896)] + [(896 + k * 9248, 896 + (k + 1) * 9248) for k in range(4)] + [(37888, 38177)]:
        assert np.abs(ref[a:b]).max() > 0
        assert np.array_equal(grad[a:b], ref[a:b]), a
