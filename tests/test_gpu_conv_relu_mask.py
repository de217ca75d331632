"""A convolution with the ReLU in its own epilogue: the signs that it keeps for the backward are those of the exact sums, and
everything behind them follows from that mask."""
import numpy as np
import pytest

import oracle
import xshinnosuke_amd as xs
from util import he_normal, rel_l2
from test_gpu_conv_split import split_everywhere
from xshinnosuke_amd.nn import functional as F

pytestmark = pytest.mark.gpu

LAYERS = [   # n c h w k r s sh sw pad
    (2, 24, 45, 61, 40, 5, 5, 1, 1, 2),      # one filter row per phase; 256-pixel tiles
    (1, 40, 16, 16, 130, 3, 3, 1, 1, 1),     # 128-pixel tiles; a row past the tile
    (3, 20, 19, 23, 70, 7, 7, 2, 2, 3),      # strided: 14 phases
    (2, 48, 14, 15, 33, 3, 3, 2, 2, 1),      # strided: four phases
    (1, 512, 7, 7, 512, 3, 3, 1, 1, 1),      # tiles that many workgroups share
    (5, 1, 25, 41, 3, 2, 2, 1, 1, 0),        # one channel, three filters
    (2, 40, 15, 17, 24, 1, 1, 1, 1, 0),      # 1 x 1
]


def _exact(x, w, sh, sw, pad):
    """The sums in float64: (K, N * OH * OW)."""
    _, col = oracle.conv2d_fwd(x, w, None, (sh, sw), pad)
    k = w.shape[0]
    return w.reshape(k, -1).astype(np.float64) @ col.astype(np.float64).T


def _layer(n, c, h, w, k, r, s, sh, sw, pad):
    rng = np.random.default_rng(n + c + k + h)
    x, wt = rng.standard_normal((n, c, h, w)).astype(np.float32), he_normal(rng, (k, c, r, s))
    oh, ow = (h + 2 * pad - r) // sh + 1, (w + 2 * pad - s) // sw + 1
    sums = _exact(x, wt, sh, sw, pad)
    assert sums.shape == (k, n * oh * ow)
    return x, wt, sums, (n, k, oh, ow)


def _flat(a):                                # (N, K, OH, OW) -> (K, N * OH * OW), the order of the kernels' pixels
    return a.transpose(1, 0, 2, 3).reshape(a.shape[1], -1)


@pytest.mark.parametrize("n,c,h,w,k,r,s,sh,sw,pad", LAYERS)
def test_signs_within_rounding_of_zero_are_the_exact_ones(gpu, n, c, h, w, k, r, s, sh, sw, pad):
    """A filter's bias takes its sum at one place away again: what is left there is half an ulp at most, and only the exact sum
    has its sign.  Two such places in every block of 32 filters by 32 pixels."""
    x, wt, sums, shape = _layer(n, c, h, w, k, r, s, sh, sw, pad)
    pixels, bias, targets = sums.shape[1], np.ones(k, np.float32), []
    for i in range(k):
        m = i % 32 // 2 * 32 + (7 * i + 3) % 32
        if m < pixels:
            bias[i] = -np.float32(sums[i, m])
            targets.append((i, m))
    want = sums + bias.astype(np.float64)[:, None] < 0
    with split_everywhere(gpu):
        args = [gpu.to_device(a) for a in (x, wt, bias)]
        mask = gpu.empty(shape, np.uint8)
        act = _flat(gpu.kernels.conv2d_fwd(*args, (sh, sw), pad, relu=True, neg_mask=mask).numpy())
        plain = _flat(gpu.kernels.conv2d_fwd(*args, (sh, sw), pad).numpy())
    mask = _flat(mask.numpy()).astype(bool)
    rows, cols = map(np.array, zip(*targets))
    np.testing.assert_array_equal(mask[rows, cols], want[rows, cols])
    np.testing.assert_array_equal(mask, want)            # and nothing else is near zero
    moved = mask != (plain < 0)
    np.testing.assert_array_equal(act[~moved], np.maximum(plain, 0)[~moved])
    exact = np.maximum(sums + bias.astype(np.float64)[:, None], 0)
    # float64 sums rounded once, and a 64-bit rounding of a partial sum below 16 for each product
    np.testing.assert_allclose(act[moved], exact[moved], rtol=2.0 ** -24, atol=c * r * s * 2.0 ** -49)
    assert not moved[np.setdiff1d(np.arange(k), rows)].any()


def test_a_block_full_of_small_sums_is_left_as_it_is(gpu):
    """More than four within rounding of zero: the block's largest sum says nothing about the others."""
    x, wt, sums, shape = _layer(*LAYERS[1])
    bias = -sums[:, 100].astype(np.float32)              # one pixel, all filters
    with split_everywhere(gpu):
        args = [gpu.to_device(a) for a in (x, wt, bias)]
        mask = gpu.empty(shape, np.uint8)
        act = gpu.kernels.conv2d_fwd(*args, (1, 1), 1, relu=True, neg_mask=mask).numpy()
        plain = gpu.kernels.conv2d_fwd(*args, (1, 1), 1).numpy()
    np.testing.assert_array_equal(_flat(act)[:128], _flat(np.maximum(plain, 0))[:128])
    np.testing.assert_array_equal(_flat(mask.numpy())[:128], _flat(plain < 0)[:128])


@pytest.mark.parametrize("n,c,h,w,k,r,pad", [(2, 24, 45, 61, 40, 5, 2), (2, 64, 28, 28, 64, 3, 1), (3, 16, 9, 7, 20, 2, 0)])
def test_the_gradients_are_those_of_the_mask(gpu, n, c, h, w, k, r, pad):
    """A sign is a decision; given it, everything else is arithmetic."""
    x, wt, sums, shape = _layer(n, c, h, w, k, r, r, 1, 1, pad)
    rng = np.random.default_rng(k)
    b, dy = (0.1 * rng.standard_normal((1, k))).astype(np.float32), rng.standard_normal(shape).astype(np.float32)
    tx, tw, tb = (xs.Tensor(gpu.to_device(a), requires_grad=True) for a in (x, wt, b))
    for _ in range(2):                                   # the second forward finds the filter's layout in place
        for t in (tx, tw, tb):
            t.zero_grad()
        y = F.conv2d(tx, tw, tb, (1, 1), pad, activation="relu")
        act, mask = y.eval.numpy(), y.cache["neg_mask"].numpy()
        y.backward(xs.Tensor(gpu.to_device(dy)))
        np.testing.assert_array_equal(_flat(mask).astype(bool), sums + b.astype(np.float64).T < 0)
        y_ref, col = oracle.conv2d_fwd(x, wt, b.reshape(-1), (1, 1), pad)
        assert rel_l2(act, np.where(mask, 0, y_ref)) <= 1e-6     # the split kernels' bound: at most 5,490 terms
        refs = oracle.conv2d_bwd(np.where(mask, 0, dy).astype(np.float32), x.shape, wt, col, (1, 1), pad, np.zeros_like(x),
                                 np.zeros_like(wt), np.zeros(k, np.float32))
        for got, want in zip((tx.grad.eval.numpy(), tw.grad.eval.numpy(), tb.grad.eval.numpy().reshape(-1)), refs):
            assert rel_l2(got, want) <= 1e-6
