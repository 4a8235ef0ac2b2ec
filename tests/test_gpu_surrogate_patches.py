"""The network's 8 x 8-pixel patches at the sizes where they can go wrong: images smaller than a
patch at every level (down to one pixel), ragged patches, and many patches, where a workgroup
takes 64 output channels and the weight gradients are split into many runs.

Against the oracle at test_gpu_surrogate's bounds (the operands' BF16 rounding).  The many-patch
case is an image tiled from a small one: the network is periodic, so its output is the small
image's tiled, bit for bit; its loss is the same mean (1e-12) and its gradient the same sum with
dY scaled by a power of two, which BF16 keeps, so only the order of FP32 sums of at most 5e5
terms differs (2e-5)."""
import numpy as np
import pytest

import surrogate_oracle as S
from cism_amd.surrogate import Surrogate
from test_gpu_surrogate import he_params, rel

pytestmark = pytest.mark.gpu


def data(rng, b, h, w):
    return (rng.standard_normal((b, h, w, 5)).astype(np.float32),
            rng.standard_normal((b, h, w, S.N_OUT)).astype(np.float32),
            (rng.random((b, h, w)) > 0.25).astype(np.float32))


@pytest.mark.parametrize("b,h,w", [(1, 8, 8), (3, 8, 40), (1, 72, 24)])
def test_small_and_ragged_images(b, h, w):
    rng = np.random.default_rng(h + w)
    th = he_params(rng)
    x, tgt, mask = data(rng, b, h, w)
    print(f"[surrogate] {b}x{h}x{w}", flush=True)
    with Surrogate(h, w, b) as net:
        net.set_params(th)
        out = net.forward(x)
        loss, g = net.loss_grad(x, tgt, mask)
    th, x, tgt, mask = (a.astype(np.float64) for a in (th, x, tgt, mask))
    assert rel(out, S.forward(th, x, bf16_ops=True)[..., :S.N_OUT]) < 5e-3
    lo, go = S.loss_grad(th, x, tgt, mask, bf16_ops=True)
    assert abs(loss - lo) <= 1e-3 * lo
    for name, wo, nw, bo, ks, ci, co, relu in S.layout()[0]:
        assert rel(g[wo:wo + nw], go[wo:wo + nw]) < 2e-2, name
        assert rel(g[bo:bo + co], go[bo:bo + co]) < 2e-2, name


def test_tiled_image():
    rng = np.random.default_rng(7)
    th = he_params(rng)
    x, tgt, mask = data(rng, 1, 64, 64)
    tile = lambda a: np.tile(a, (2, 4, 4) + (1,) * (a.ndim - 3))   # noqa: E731
    got = []
    for n, args in ((1, (x, tgt, mask)), (2, tuple(tile(a) for a in (x, tgt, mask)))):
        with Surrogate(64 if n == 1 else 256, 64 if n == 1 else 256, n) as net:
            net.set_params(th)
            got.append((net.forward(args[0]),) + net.loss_grad(*args))
    (o1, l1, g1), (o2, l2, g2) = got
    assert np.array_equal(o2, tile(o1))
    assert abs(l2 - l1) <= 1e-12 * l1
    assert rel(g2, g1.astype(np.float64)) < 2e-5
