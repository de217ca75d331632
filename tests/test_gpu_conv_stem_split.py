"""First layers (1 or 3 channels, stride 2) on split operands: against the oracle at the edges of tiles, rows and images.

Bound: as for the other split kernels, at most 2^-24 of each term is dropped and sums of at most 147 terms are float32:
1e-6 in relative L2 norm is far above rounding and far below any misplaced term."""
import numpy as np
import pytest

import oracle
from util import he_normal, rel_l2

pytestmark = pytest.mark.gpu
TOL = 1e-6


def _fp32_kernel(gpu, x, w, b, pad):
    """The same by the kernel on the fp32 matrix instructions, whose sums have another order."""
    old = gpu.set_option("conv_split", 0)
    try:
        return gpu.kernels.conv2d_fwd(x, w, b, (2, 2), pad).numpy()
    finally:
        gpu.set_option("conv_split", old)


@pytest.mark.parametrize("n,c,h,w,k,r,pad", [
    (1, 3, 64, 64, 64, 7, 3),        # one wide tile across, four down
    (2, 3, 63, 65, 32, 7, 3),        # a pixel past the tile, half of the filters
    (3, 3, 32, 32, 65, 7, 3),        # square tiles; a filter past the row tile
    (2, 3, 40, 41, 36, 7, 3),        # the last rows in one half of the lanes only
    (1, 3, 7, 200, 64, 7, 0),        # one row of outputs, 97 across
    (5, 3, 224, 31, 40, 7, 2),       # narrow images
    (40, 3, 64, 48, 128, 7, 3),      # more tiles than workgroups, two row tiles
    (9, 3, 97, 113, 33, 5, 2),
    (2, 3, 50, 34, 64, 5, 0),
    (4, 3, 65, 33, 96, 3, 1),
    (3, 3, 33, 32, 64, 3, 5),        # a border wider than the filter
    (3, 1, 61, 97, 48, 7, 3),        # one channel: the last filter row by itself
    (5, 1, 30, 29, 65, 7, 0),
    (130, 1, 28, 28, 32, 7, 3),      # ... more tiles than workgroups
])
def test_first_layer_against_the_oracle(gpu, n, c, h, w, k, r, pad):
    K = gpu.kernels
    rng = np.random.default_rng(n + 5 * h + k)
    x = rng.standard_normal((n, c, h, w)).astype(np.float32)
    wt, b = he_normal(rng, (k, c, r, r)), rng.standard_normal((k,)).astype(np.float32)
    y_ref, _ = oracle.conv2d_fwd(x, wt, b, (2, 2), pad)
    dx, dw, db = (gpu.to_device(a) for a in (x, wt, b))
    y = K.conv2d_fwd(dx, dw, db, (2, 2), pad).numpy()
    assert rel_l2(y, y_ref) <= TOL
    assert (y != _fp32_kernel(gpu, dx, dw, db, pad)).any()
    mask = gpu.empty(y.shape, np.uint8)
    act = K.conv2d_fwd(dx, dw, db, (2, 2), pad, relu=True, neg_mask=mask).numpy()
    np.testing.assert_array_equal(act, np.maximum(y, 0.0))
    np.testing.assert_array_equal(mask.numpy(), (y < 0).astype(np.uint8))


@pytest.mark.parametrize("c,h,w,r,pad", [(3, 40, 44, 7, 3), (1, 33, 66, 7, 2), (3, 31, 70, 5, 2), (3, 45, 33, 3, 1)])
def test_values_that_do_not_split(gpu, c, h, w, r, pad):
    """Infinities, NaN, the largest floats and values near the smallest: sums are what the fp32 kernels give, and no value
    reaches a sum whose window it is not in."""
    K = gpu.kernels
    rng = np.random.default_rng(c)
    x = (rng.standard_normal((3, c, h, w)) * 0.1).astype(np.float32)
    wt = he_normal(rng, (40, c, r, r))
    x[0, 0, 5, 9], x[1, c - 1, h - 1, w - 1], x[1, 0, 0, 0] = np.inf, np.nan, np.float32(3.4e38)
    wt[3, 0, 0, 1], wt[7, c - 1, r - 1, r - 1] = -np.inf, np.nan
    x[2] *= np.float32(2.0 ** -120)
    dx, dw = gpu.to_device(x), gpu.to_device(wt)
    got = K.conv2d_fwd(dx, dw, None, (2, 2), pad).numpy()
    plain = _fp32_kernel(gpu, dx, dw, None, pad)
    for test in (np.isnan, np.isposinf, np.isneginf):
        np.testing.assert_array_equal(test(got), test(plain))
    calm = np.isfinite(plain[:2])
    assert calm.any() and not calm.all() and rel_l2(got[:2][calm], plain[:2][calm]) <= TOL
    assert (got[:2][calm] != plain[:2][calm]).any()
    good = [i for i in range(40) if i not in (3, 7)]
    y_ref, _ = oracle.conv2d_fwd(x[2:].astype(np.float64) * 2.0 ** 120, wt[good], np.zeros(len(good), np.float32), (2, 2), pad)
    assert rel_l2(got[2:, good].astype(np.float64) * 2.0 ** 120, y_ref) <= 1e-5      # sums near the smallest normal float


def test_a_workspace_without_room_for_a_copy(gpu):
    """The kernel reads image and filter themselves: the size that the library asks for has no copy of the input (20 MB here), and
    that size, or the static buffer of the forward that takes none, gives the same bits."""
    from xshinnosuke_amd.backend import capi
    K = gpu.kernels
    rng = np.random.default_rng(3)
    dims = (32, 3, 224, 224, 64, 7, 7, 2, 2, 3)
    x, w = gpu.to_device(rng.standard_normal(dims[:4]).astype(np.float32)), gpu.to_device(he_normal(rng, (64, 3, 7, 7)))
    want = K.conv2d_fwd(x, w, None, (2, 2), 3).numpy()
    size = capi.lib.raw("xsmi_conv2d_pass_workspace_bytes")(*dims, 0, 0)
    assert size < 1 << 20
    ws, y = gpu.empty(((size + 3) // 4,)), gpu.empty(want.shape)
    capi.lib.call("xsmi_conv2d_fwd", x.ptr, w.ptr, None, y.ptr, None, *dims, 0, ws.ptr, size)
    np.testing.assert_array_equal(y.numpy(), want)
    z = gpu.empty(want.shape)
    capi.lib.call("xsmi_conv2d_fwd_noalloc", x.ptr, w.ptr, None, z.ptr, None, *dims, 0)
    np.testing.assert_array_equal(z.numpy(), want)


@pytest.mark.parametrize("n,c,h,w,k,r,pad,split", [
    (244, 1, 12, 12, 177, 7, 0, False),      # 9 outputs in a tile of 256, three row tiles
    (210, 3, 14, 9, 186, 7, 0, False),
    (77, 1, 56, 21, 240, 7, 3, False),       # 0.60 full
    (28, 1, 12, 12, 177, 7, 0, True),        # the same in 84 tiles
    (70, 3, 54, 54, 128, 7, 3, True),        # 27 x 27 outputs: 0.71 full
])
def test_images_that_leave_their_tiles_empty_go_to_the_fp32_kernel(gpu, n, c, h, w, k, r, pad, split):
    """Where there are more tiles than compute units it was up to twice as fast there; the bits tell the kernels apart."""
    rng = np.random.default_rng(k)
    x, wt = gpu.to_device(rng.standard_normal((n, c, h, w)).astype(np.float32)), gpu.to_device(he_normal(rng, (k, c, r, r)))
    got, plain = gpu.kernels.conv2d_fwd(x, wt, None, (2, 2), pad).numpy(), _fp32_kernel(gpu, x, wt, None, pad)
    assert rel_l2(got, plain) <= TOL
    assert (got != plain).any() == split
