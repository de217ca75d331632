"""The fp32 convolution on bf16 matrix pipes (three-way split operands): every geometry it serves against the oracle,
at the edges of its tiles, channel groups, phases and grids.

Bound: the split drops at most 2^-24 of each term and adds in float32; the worst of the sizes here, 4608 terms,
was 1.7e-7 in relative L2 norm, so 1e-6 is far above rounding and far below any misplaced term."""
import contextlib

import numpy as np
import pytest

import oracle
from util import he_normal, rel_l2, round_bf16

pytestmark = pytest.mark.gpu
TOL = 1e-6


@contextlib.contextmanager
def split_everywhere(gpu):
    old = gpu.set_option("conv_split", 2)
    try:
        yield
    finally:
        gpu.set_option("conv_split", old)


def _data(n, c, h, w, k, r, s, sh, sw, pad, gpu):
    rng = np.random.default_rng(n + 3 * c + 7 * k + h)
    oh, ow = gpu.kernels.conv_out_hw(h, w, r, s, (sh, sw), pad)
    return (rng.standard_normal((n, c, h, w)).astype(np.float32), he_normal(rng, (k, c, r, s)),
            rng.standard_normal((k,)).astype(np.float32), rng.standard_normal((n, k, oh, ow)).astype(np.float32),
            rng.standard_normal((n, c, h, w)).astype(np.float32))


@pytest.mark.parametrize("n,c,h,w,k,r,s,sh,sw,pad", [
    (1, 16, 1, 255, 64, 1, 3, 1, 1, 1),      # one row tile, one pixel short of two 128-pixel tiles
    (1, 17, 16, 16, 65, 3, 3, 1, 1, 1),      # 256 pixels; a channel and a row past their tiles
    (1, 31, 11, 93, 63, 3, 3, 1, 1, 1),      # 1023 pixels: the last of the narrow tiles
    (1, 33, 32, 32, 1, 3, 3, 1, 1, 1),       # 1024: the first of the wide ones; one row
    (5, 1, 25, 41, 3, 2, 2, 1, 1, 0),        # one channel, even filter, no padding
    (3, 32, 9, 3, 64, 3, 3, 1, 1, 1),        # rows of three pixels: many row and image ends in a tile
    (2, 24, 45, 61, 40, 5, 5, 1, 1, 2),      # an image does not hold all rows' taps: one filter row per phase
    (3, 20, 19, 23, 70, 7, 7, 2, 2, 3),      # strided, one filter row per phase: 14 phases
    (2, 48, 14, 15, 20, 3, 3, 2, 2, 1),      # four phases forward, four classes backward
    (2, 20, 17, 13, 70, 3, 5, 2, 1, 1),      # strides and filter sides that differ
    (2, 40, 15, 17, 24, 1, 1, 1, 1, 0),      # 1 x 1: one step per channel group
    (2, 18, 12, 12, 24, 3, 3, 3, 3, 0),      # stride 3: nine phases of one tap
    (1, 512, 7, 7, 512, 3, 3, 1, 1, 1),      # every tile shared by many workgroups
    (20, 32, 56, 56, 64, 3, 3, 1, 1, 1),     # more tiles than workgroups
    (20, 64, 45, 57, 32, 3, 3, 1, 1, 1),     # few rows: tiles of 32 x 512, the last one 100 pixels
    (17, 31, 56, 56, 1, 5, 5, 1, 1, 2),      # the same with two images for five filter rows, one row
    (11, 17, 61, 70, 33, 7, 7, 1, 1, 3),     # a row past them: 64 x 256, images of 3, 3 and 1 filter rows
    (24, 33, 56, 57, 20, 5, 5, 2, 2, 2),     # few rows, strided: 28 x 29 outputs, backward-data of four classes
    (17, 98, 57, 57, 97, 3, 3, 2, 2, 1),     # strided, 128 x 128: seven groups, the last of one or two channels
    (34, 200, 29, 28, 96, 3, 3, 2, 2, 0),    # two row tiles backward, the second of 72 rows; images of 6, 4, 4 and 2 groups
    (9, 80, 112, 113, 200, 3, 3, 2, 2, 1),   # rows of 57 pixels: three of the four phases in one image
    (7, 96, 56, 130, 128, 2, 4, 2, 3, 1),    # filter sides and strides that differ
    (1, 40, 28, 37, 130, 3, 3, 1, 1, 1),     # tiles with workgroups of their own: 1036 pixels, two rows past two tiles
    (2, 100, 9, 9, 24, 5, 5, 2, 2, 2),       # ... in classes of 9, 6, 6 and 4 taps, shared by different numbers of them
    (8, 16, 40, 40, 10, 3, 3, 1, 1, 1),      # ... one for each
])
def test_split_convolution_against_the_oracle(gpu, n, c, h, w, k, r, s, sh, sw, pad):
    K = gpu.kernels
    x, wt, b, dy, dx0 = _data(n, c, h, w, k, r, s, sh, sw, pad, gpu)
    y_ref, col = oracle.conv2d_fwd(x, wt, b, (sh, sw), pad)
    dx_ref, _, _ = oracle.conv2d_bwd(dy, x.shape, wt, col, (sh, sw), pad, dx0.copy(), np.zeros_like(wt), np.zeros_like(b))
    dx_, dw_, db_, ddy = (gpu.to_device(a) for a in (x, wt, b, dy))
    with split_everywhere(gpu):
        y = K.conv2d_fwd(dx_, dw_, db_, (sh, sw), pad).numpy()
        assert rel_l2(y, y_ref) <= TOL
        mask = gpu.empty(y.shape, np.uint8)
        act = K.conv2d_fwd(dx_, dw_, db_, (sh, sw), pad, relu=True, neg_mask=mask).numpy()
        np.testing.assert_array_equal(act, np.maximum(y, 0.0))
        np.testing.assert_array_equal(mask.numpy(), (y < 0).astype(np.uint8))
        gx = gpu.to_device(dx0)
        K.conv2d_bwd_data(ddy, dw_, x.shape, (sh, sw), pad, dx=gx, accumulate=True)
        assert rel_l2(gx.numpy(), dx_ref) <= TOL


@pytest.mark.parametrize("n,c,h,w,k,pad", [
    (1, 3, 3, 3, 2, 0),                      # one output pixel
    (2, 65, 7, 8, 63, 1),                    # a channel past an octet, a filter short of a tile
    (3, 16, 5, 9, 64, 1),                    # 45 pixels: two images end inside a stage
    (2, 64, 6, 7, 64, 0),                    # no padding
    (3, 20, 11, 17, 70, 0),                  # no padding, few filters past two tiles of 32
    (9, 64, 14, 14, 128, 1),                 # uneven splits
    (2, 130, 56, 56, 64, 1),                 # twenty splits: four waves share them
    (40, 96, 14, 15, 200, 1),                # nine splits
])
@pytest.mark.parametrize("accumulate", [False, True])
def test_split_weight_gradient_against_the_oracle(gpu, n, c, h, w, k, pad, accumulate):
    K = gpu.kernels
    x, wt, b, dy, _ = _data(n, c, h, w, k, 3, 3, 1, 1, pad, gpu)
    dw0, db0 = (wt, b) if accumulate else (np.zeros_like(wt), np.zeros_like(b))
    _, col = oracle.conv2d_fwd(x, wt, b, (1, 1), pad)
    _, dw_ref, db_ref = oracle.conv2d_bwd(dy, x.shape, wt, col, (1, 1), pad, np.zeros_like(x), dw0.copy(), db0.copy())
    gw, gb = gpu.to_device(dw0), gpu.to_device(db0)
    with split_everywhere(gpu):
        K.conv2d_bwd_weight(gpu.to_device(dy), gpu.to_device(x), wt.shape, (1, 1), pad, dw=gw, db=gb, accumulate=accumulate)
    assert rel_l2(gw.numpy(), dw_ref) <= TOL and rel_l2(gb.numpy(), db_ref) <= TOL


@pytest.mark.parametrize("n,c,h,w,k,r,s,sh,sw,pad", [
    (1, 3, 3, 3, 2, 3, 3, 1, 1, 0),          # one output pixel; an octet of three channels
    (2, 65, 7, 8, 63, 3, 3, 1, 1, 1),        # a channel past an octet, a filter short of a tile
    (3, 20, 19, 23, 70, 7, 7, 2, 2, 3),      # strided, few filters past a tile of 64
    (2, 20, 17, 13, 33, 3, 5, 2, 1, 1),      # strides and filter sides that differ
    (2, 40, 15, 17, 24, 1, 1, 2, 2, 0),      # one tap across: slots are the columns that are read
    (2, 18, 12, 12, 24, 2, 2, 3, 3, 0),      # columns between the taps
    (1, 8, 20, 40, 130, 15, 16, 1, 1, 7),    # the widest filter that is served but one
    (7, 5, 9, 1, 40, 3, 1, 2, 1, 1),         # one input column: rows of three slots
    (4, 24, 5, 4, 40, 5, 5, 1, 1, 2),        # rows of four pixels, many row and image ends in a stage
    (2, 24, 1, 70, 16, 1, 7, 1, 1, 3),       # one row, padding above and below it only
    (3, 96, 9, 9, 8, 3, 3, 1, 1, 2),         # more padding than the filter needs
    (9, 64, 14, 14, 128, 3, 3, 1, 1, 1),     # uneven splits
    (40, 96, 14, 15, 200, 3, 3, 2, 2, 1),    # nine splits: four waves share them
    (2, 12, 60, 60, 24, 5, 5, 1, 1, 2),      # 113 splits: sixteen waves
    (1, 8, 3, 2700, 8, 1, 3, 1, 1, 0),       # rows that 24-bit division does not hold: the fp32 kernels
])
def test_split_weight_gradient_of_any_filter(gpu, n, c, h, w, k, r, s, sh, sw, pad):
    """Against the oracle, with ordinary values, and with values that are not finite in both operands: the workgroups that meet
    them form their sums again."""
    K = gpu.kernels
    x, wt, b, dy, _ = _data(n, c, h, w, k, r, s, sh, sw, pad, gpu)
    for finite in (True, False):
        if not finite:
            x[-1, c // 2, h // 2, w // 2] = np.nan
            dy[0, k // 2, dy.shape[2] // 2, -1] = np.inf
        _, col = oracle.conv2d_fwd(x, wt, b, (sh, sw), pad)
        with np.errstate(all="ignore"):
            _, ref, db_ref = oracle.conv2d_bwd(dy, x.shape, wt, col, (sh, sw), pad, np.zeros_like(x), np.zeros_like(wt), np.zeros_like(b))
        with split_everywhere(gpu):
            gw, gb = K.conv2d_bwd_weight(gpu.to_device(dy), gpu.to_device(x), wt.shape, (sh, sw), pad, want_db=True)
        for got, want in ((gw.numpy(), ref), (gb.numpy(), db_ref)):
            for test in (np.isnan, np.isposinf, np.isneginf):
                np.testing.assert_array_equal(test(got), test(want))
            calm = np.isfinite(want)
            assert not calm.any() or rel_l2(got[calm], want[calm]) <= TOL


@pytest.mark.parametrize("tile,dims", [    # filters, pixels of a stage, pairs of units, rounds of staging; a layer that fills it
    (646422, (2, 20, 11, 13, 70, 3, 2, 1, 1, 1)), (646423, (2, 130, 11, 13, 40, 3, 1, 2, 2, 1)),
    (646432, (2, 20, 11, 13, 40, 7, 7, 2, 2, 3)), (646433, (2, 20, 11, 13, 70, 3, 3, 2, 2, 1)),
    (646442, (2, 20, 9, 26, 40, 5, 5, 1, 1, 2)), (646443, (2, 20, 11, 13, 40, 5, 5, 1, 1, 2)),
    (646452, (2, 20, 9, 26, 40, 5, 5, 1, 1, 2)), (646453, (2, 20, 11, 13, 40, 7, 7, 2, 2, 3)),
    (643222, (2, 20, 11, 13, 70, 3, 2, 3, 3, 1)), (643223, (2, 20, 11, 13, 70, 3, 2, 3, 3, 1)),
    (643232, (2, 20, 11, 13, 70, 3, 3, 2, 2, 1)), (643233, (2, 41, 11, 13, 70, 3, 2, 3, 3, 1)),
    (643242, (2, 41, 11, 13, 70, 3, 3, 2, 2, 1)), (643243, (2, 130, 11, 13, 40, 5, 1, 1, 1, 2)),
    (643252, (2, 130, 11, 13, 40, 3, 2, 1, 1, 1)), (643253, (2, 90, 11, 13, 40, 3, 3, 2, 2, 1)),
    (326422, (2, 20, 11, 13, 70, 3, 3, 1, 1, 1)), (326423, (2, 130, 11, 13, 40, 3, 2, 1, 1, 1)),
    (326432, (2, 20, 11, 13, 40, 5, 5, 1, 1, 2)), (326433, (2, 20, 11, 13, 40, 7, 7, 2, 2, 3)),
    (326442, (2, 20, 9, 26, 40, 7, 7, 1, 1, 3)), (326443, (2, 90, 11, 13, 40, 5, 5, 1, 1, 2)),
    (326452, (2, 20, 9, 26, 40, 7, 7, 1, 1, 3)), (326453, (2, 130, 9, 26, 40, 5, 5, 1, 1, 2)),
    (323222, (2, 20, 11, 13, 70, 3, 3, 2, 2, 1)), (323223, (2, 130, 11, 13, 40, 3, 2, 3, 3, 1)),
    (323232, (2, 20, 11, 13, 40, 7, 7, 2, 2, 3)), (323233, (2, 130, 11, 13, 40, 3, 3, 2, 2, 1)),
    (323242, (2, 20, 11, 13, 40, 7, 7, 2, 2, 3)), (323243, (2, 41, 15, 8, 40, 7, 7, 2, 2, 3)),
    (323252, (2, 41, 9, 26, 40, 7, 7, 2, 2, 3)), (323253, (2, 41, 11, 13, 40, 7, 7, 2, 2, 3)),
])
def test_split_weight_gradient_of_every_tile(gpu, tile, dims):
    """Each instantiation against the oracle: ordinary values, every sum formed again (powers of two are exact), and values that
    are not finite in both operands."""
    n, c, h, w, k, r, s, sh, sw, pad = dims
    x, wt, b, dy, _ = _data(*dims, gpu)
    run = lambda: gpu.kernels.conv2d_bwd_weight(gpu.to_device(dy), gpu.to_device(x), wt.shape, (sh, sw), pad, want_db=True)  # noqa: E731
    old = gpu.set_option("conv_split", 0)
    try:
        fp32 = run()[0].numpy()
    finally:
        gpu.set_option("conv_split", old)
    gpu.set_option("wgrad_tile", tile)
    try:
        with split_everywhere(gpu):
            for values in ("ordinary", "small", "not finite"):
                if values == "small":
                    x, scale = x * np.float32(2.0 ** -107), 2.0 ** 107
                elif values == "not finite":
                    x, scale = x * np.float32(2.0 ** 107), 1.0
                    x[-1, c // 2, h // 2, w // 2], dy[0, k // 2, dy.shape[2] // 2, -1] = np.nan, np.inf
                else:
                    scale = 1.0
                _, col = oracle.conv2d_fwd(x * np.float32(scale), wt, b, (sh, sw), pad)
                with np.errstate(all="ignore"):
                    _, ref, db_ref = oracle.conv2d_bwd(dy, x.shape, wt, col, (sh, sw), pad, np.zeros_like(x), np.zeros_like(wt), np.zeros_like(b))
                gw, gb = (a.numpy() for a in run())
                assert values != "ordinary" or not np.array_equal(gw, fp32)      # a tile that does not fit leaves the call to them
                for got, want in ((gw.astype(np.float64) * scale, ref), (gb, db_ref)):
                    for test in (np.isnan, np.isposinf, np.isneginf):
                        np.testing.assert_array_equal(test(got), test(want))
                    calm = np.isfinite(want)
                    assert not calm.any() or rel_l2(got[calm], want[calm]) <= TOL
    finally:
        gpu.set_option("wgrad_tile", 0)


@pytest.mark.parametrize("w,pad", [(56, 1), (7, 1)])       # a stage is 64 pixels: little more than a row, nine rows
@pytest.mark.parametrize("relu", [False, True])
def test_weight_gradient_rounds_to_both_sides(gpu, w, pad, relu):
    """The bf16 MFMA drops what small products have below an accumulator's last bits, always downwards; over the two halves of a
    workgroup that cancels.  4,608 errors of one sign have a mean next to their rms, independent ones 1/68 of it: ten times
    that.  And the error against 64 bits is no larger than that of the fp32 kernels."""
    n, c, h, k, part = 8 * 56 // w, 64, 56, 512, 8
    rng = np.random.default_rng(w)
    x = rng.standard_normal((n, c, h, w)).astype(np.float32)
    x = np.maximum(x, 0) if relu else x
    dy = rng.standard_normal((n, k, h, w)).astype(np.float32)
    xp = np.pad(x, ((0, 0), (0, 0), (1, 1), (1, 1))).astype(np.float64)
    d = dy[:, :part].astype(np.float64).transpose(1, 0, 2, 3).reshape(part, -1)
    ref = np.stack([d @ xp[:, :, r:r + h, s:s + w].transpose(0, 2, 3, 1).reshape(-1, c) for r in range(3) for s in range(3)], 2)
    errors = {}
    for option in (2, 0):
        old = gpu.set_option("conv_split", option)
        try:
            got = gpu.kernels.conv2d_bwd_weight(gpu.to_device(dy), gpu.to_device(x), (k, c, 3, 3), (1, 1), pad)[0].numpy()
        finally:
            gpu.set_option("conv_split", old)
        errors[option] = got[:part].reshape(part, c, 9).astype(np.float64) - ref
    rms = {o: np.sqrt((e ** 2).mean()) for o, e in errors.items()}
    assert abs(errors[2].mean()) <= 0.147 * rms[2]
    assert rms[2] <= rms[0]


@pytest.mark.parametrize("n,h,w,r,stride,pad,products", [      # at most, for an element of the gradient
    (1, 1, 1, 3, 1, 1, 1), (1, 2, 2, 7, 2, 3, 1), (1, 7, 7, 7, 1, 0, 1), (1, 1, 2, 5, 1, 2, 2), (2, 1, 1, 3, 2, 1, 2), (1, 1, 3, 5, 1, 2, 3),
    (1, 2, 2, 3, 1, 1, 4), (1, 3, 3, 7, 2, 3, 4),              # the last that are formed in float64
    (3, 1, 1, 3, 1, 1, 3), (2, 1, 2, 3, 1, 1, 4), (1, 3, 3, 3, 1, 1, 9), (1, 1, 8, 5, 1, 2, 8)])
def test_weight_gradient_of_a_few_products(gpu, n, h, w, r, stride, pad, products):
    """One product is rounded once, to nearest; a few are no further from 64 bits than the fp32 kernels' sums."""
    c, k = 64, 96
    rng = np.random.default_rng(n + h + w + r)
    oh, ow = gpu.kernels.conv_out_hw(h, w, r, r, (stride, stride), pad)
    x, dy = rng.standard_normal((n, c, h, w)).astype(np.float32), rng.standard_normal((n, k, oh, ow)).astype(np.float32)
    xp = np.pad(x, ((0, 0), (0, 0), (pad, pad), (pad, pad))).astype(np.float64)
    taps = [[xp[:, :, a:a + oh * stride:stride, b:b + ow * stride:stride] for b in range(r)] for a in range(r)]
    assert max(int((t != 0).sum(axis=(0, 2, 3)).max()) for row in taps for t in row) == products
    ref = np.stack([np.stack([np.einsum("nkhw,nchw->kc", dy.astype(np.float64), t) for t in row], 2) for row in taps], 2)
    run = lambda: gpu.kernels.conv2d_bwd_weight(gpu.to_device(dy), gpu.to_device(x), (k, c, r, r), (stride, stride), pad)[0].numpy()  # noqa: E731
    got = run()
    old = gpu.set_option("conv_split", 0)
    try:
        fp32 = run()
    finally:
        gpu.set_option("conv_split", old)
    assert rel_l2(got, ref) <= rel_l2(fp32, ref)
    if products == 1:
        np.testing.assert_array_equal(got, ref.astype(np.float32))


FORMED_AGAIN = [   # what the kernel that forms sums again walks differently
    (1, 17, 16, 16, 65, 3, 3, 1, 1, 1),      # a channel and a row past their tiles
    (5, 1, 25, 41, 3, 2, 2, 1, 1, 0),        # one channel, even filter
    (2, 24, 45, 61, 40, 5, 5, 1, 1, 2),      # one filter row per phase
    (3, 20, 19, 23, 70, 7, 7, 2, 2, 3),      # strided: 14 phases
    (2, 48, 14, 15, 20, 3, 3, 2, 2, 1),      # four phases forward, four classes backward
    (2, 20, 17, 13, 70, 3, 5, 2, 1, 1),      # strides and filter sides that differ
    (1, 512, 7, 7, 512, 3, 3, 1, 1, 1),      # segments that begin and end anywhere in a tile
    (17, 31, 56, 56, 31, 5, 5, 1, 1, 2),     # tiles of 32 x 512 in both passes, two images for five filter rows
    (24, 33, 56, 57, 20, 5, 5, 2, 2, 2),     # 32 x 512 forward and strided
    (17, 98, 57, 57, 97, 3, 3, 2, 2, 1),     # 128 x 128: images of several phases or channel groups
]


@pytest.mark.parametrize("n,c,h,k,st,split", [
    (32, 64, 32, 128, 2, False),             # 256 tiles of a data gradient by taps: the most that leave a compute unit
    (33, 64, 32, 128, 2, True),              # 264: the data gradient fills the chip
    (20, 64, 28, 256, 2, True),              # four times as many filters as channels
    (8, 128, 28, 128, 1, False),             # a split data gradient of few tiles: in order, 9.2e8 products
    (16, 128, 28, 128, 1, True),             # 1.8e9
    (32, 512, 7, 512, 1, True),
    (42, 256, 14, 128, 1, True),             # 260 tiles
    (5, 64, 56, 255, 1, True),               # no bf16 kernel for 255 filters, so no bf16 data gradient to let in
])
def test_weight_gradient_beside_a_bf16_data_gradient(gpu, n, c, h, k, st, split):
    """A bf16 data gradient by taps that leaves compute units idle runs beside the weight gradient, whose split form would keep
    it out of them; before a split one few products run on the tap kernel.  One call for both gradients and one for each give
    the same bits."""
    K = gpu.kernels
    rng = np.random.default_rng(h)
    x, w, dy = (gpu.to_device(rng.standard_normal(s).astype(np.float32)) for s in ((n, c, h, h), (k, c, 3, 3), (n, k, h // st, h // st)))
    own = K.conv2d_bwd_weight(dy, x, w.shape, (st, st), 1, bf16=True)[0].numpy()
    dw = gpu.empty(w.shape)
    K.conv2d_bwd(dy, x, w, gpu.empty(x.shape), dw, None, (st, st), 1, bf16=True)
    np.testing.assert_array_equal(dw.numpy(), own)
    old = gpu.set_option("conv_split", 0)
    try:
        fp32 = K.conv2d_bwd_weight(dy, x, w.shape, (st, st), 1)[0].numpy()
    finally:
        gpu.set_option("conv_split", old)
    assert np.array_equal(own, fp32) is not split


@pytest.mark.parametrize("n,c,h,w,k,r,s,sh,sw,pad", FORMED_AGAIN)
def test_sums_that_are_formed_again(gpu, n, c, h, w, k, r, s, sh, sw, pad):
    """Every sum is below 2^-100, so every one is formed a second time; powers of two are exact: the bound is that of
    ordinary values."""
    K = gpu.kernels
    x, wt, b, dy, _ = _data(n, c, h, w, k, r, s, sh, sw, pad, gpu)
    y_ref, col = oracle.conv2d_fwd(x, wt, 0 * b, (sh, sw), pad)
    dx_ref, _, _ = oracle.conv2d_bwd(dy, x.shape, wt, col, (sh, sw), pad, np.zeros_like(x), np.zeros_like(wt), np.zeros_like(b))
    small = lambda a: gpu.to_device(a * np.float32(2.0 ** -107))  # noqa: E731
    with split_everywhere(gpu):
        y = K.conv2d_fwd(small(x), gpu.to_device(wt), None, (sh, sw), pad).numpy()
        gx = K.conv2d_bwd_data(small(dy), gpu.to_device(wt), x.shape, (sh, sw), pad).numpy()
    assert rel_l2(y.astype(np.float64) * 2.0 ** 107, y_ref) <= TOL and rel_l2(gx.astype(np.float64) * 2.0 ** 107, dx_ref) <= TOL


@pytest.mark.parametrize("pass_", [0, 1])
def test_a_filter_whose_layout_is_in_place_is_not_read(gpu, pass_):
    """What is passed as the filter is another one by then; a value that does not split, on either side, takes the sums that
    are formed again, and those take the filter from its layout too."""
    import ctypes
    from xshinnosuke_amd.backend import capi
    dims = (2, 40, 12, 13, 40, 3, 3, 1, 1, 1)
    x, wt, _, _, _ = _data(*dims, gpu)
    x[:, [2, 33]] *= np.float32(0.1)                     # products with 3.4e38 stay finite in 32 bits as well
    x[0, 3, 2, 2], x[1, 19, 6, 6], x[1, 20, 11, 12] = np.inf, np.nan, np.float32(3.4e38)
    wt[5, 3, 0, 2], wt[7, 30, 1, 1], wt[33, 2, 2, 0] = -np.inf, np.nan, np.float32(-3.4e38)
    K = gpu.kernels
    run = lambda: (K.conv2d_bwd_data(dx, dw, x.shape, (1, 1), 1) if pass_ else K.conv2d_fwd(dx, dw, None, (1, 1), 1)).numpy()  # noqa: E731
    dx, dw, other = gpu.to_device(x), gpu.to_device(wt), gpu.to_device(np.ones_like(wt))
    with split_everywhere(gpu):
        ref = run()
        size = capi.lib.raw("xsmi_conv2d_pass_workspace_bytes")(*dims, pass_, 0)
        ws, y = gpu.empty(((size + 3) // 4,)), gpu.empty(ref.shape)
        job = (capi.PackJob * 1)()
        job[0].w, job[0].workspace, job[0].workspace_bytes = dw.ptr, ws.ptr, size
        for field, v in zip(("N", "C", "H", "W", "K", "R", "S", "sh", "sw", "pad", "pass_"), dims + (pass_,)):
            setattr(job[0], field, v)
        capi.lib.call("xsmi_conv2d_pack", 1, ctypes.cast(job, ctypes.c_void_p))
        capi.lib.call("xsmi_conv2d_bwd_join")
        assert job[0].packed == 1
        if pass_ == 0:
            capi.lib.call("xsmi_conv2d_fwd", dx.ptr, other.ptr, None, y.ptr, None, *dims, capi.CONV_WS_PACKED, ws.ptr, size)
        else:
            capi.lib.call("xsmi_conv2d_bwd_data", dx.ptr, other.ptr, y.ptr, *dims, 0.0, capi.CONV_WS_PACKED, ws.ptr, size)
    got = y.numpy()
    assert got.tobytes() == ref.tobytes()
    old = gpu.set_option("conv_split", 0)
    try:
        plain = run()
    finally:
        gpu.set_option("conv_split", old)
    for test in (np.isnan, np.isposinf, np.isneginf):
        np.testing.assert_array_equal(test(got), test(plain))
    calm = np.isfinite(plain)
    assert calm.any() and rel_l2(got[calm], plain[calm]) <= TOL


@pytest.mark.parametrize("n,c,h,w,k,r,s,sh,sw,pad", [
    (1, 64, 1, 255, 32, 1, 3, 1, 1, 1),      # one pixel short of two 128-pixel tiles
    (1, 65, 16, 16, 64, 3, 3, 1, 1, 1),      # a row past the tile
    (3, 17, 32, 32, 96, 3, 3, 1, 1, 0),      # wide tiles
    (2, 40, 45, 61, 32, 5, 5, 1, 1, 2),      # an image does not hold all rows' taps
    (1, 512, 7, 7, 512, 3, 3, 1, 1, 1),      # every tile shared by many workgroups
    (20, 64, 56, 56, 32, 3, 3, 1, 1, 1),     # more tiles than workgroups
    (20, 16, 45, 57, 64, 3, 3, 1, 1, 1),     # few rows: tiles of 32 x 512
    (34, 96, 29, 28, 224, 3, 3, 2, 2, 0),    # strided, 128 x 128
    (2, 24, 19, 23, 64, 7, 7, 2, 2, 3),      # four classes
    (2, 18, 13, 12, 32, 2, 2, 2, 2, 0),      # four of one tap
    (3, 18, 12, 14, 32, 4, 3, 2, 1, 1),      # two
    (2, 30, 15, 17, 64, 1, 1, 1, 1, 0),
    (13, 98, 57, 57, 64, 2, 2, 1, 1, 1),
])
def test_bf16_data_gradient(gpu, n, c, h, w, k, r, s, sh, sw, pad):
    """On operands rounded to bf16 only the float32 sums differ from the oracle's: 1e-5, as for the other bf16 kernels.  What
    is not finite is so where it is with the kernel that gathers dy tap by tap."""
    K = gpu.kernels
    x, wt, b, dy, dx0 = _data(n, c, h, w, k, r, s, sh, sw, pad, gpu)
    _, col = oracle.conv2d_fwd(x, round_bf16(wt), b, (sh, sw), pad)
    ref, _, _ = oracle.conv2d_bwd(round_bf16(dy), x.shape, round_bf16(wt), col, (sh, sw), pad, dx0.copy(), np.zeros_like(wt), np.zeros_like(b))
    dw_, ddy, gx = gpu.to_device(wt), gpu.to_device(dy), gpu.to_device(dx0)
    with split_everywhere(gpu):
        K.conv2d_bwd_data(ddy, dw_, x.shape, (sh, sw), pad, dx=gx, accumulate=True, bf16=True)
    assert rel_l2(gx.numpy(), ref) <= 1e-5
    dy[0, 1, 0, 0], dy[-1, -1, -1, -1], dy[0, 0, -1, -1] = np.inf, np.nan, np.float32(3.4e38)
    wt[0, -1, 0, 0] = -np.inf
    dw_, ddy = gpu.to_device(wt), gpu.to_device(dy)
    run = lambda: K.conv2d_bwd_data(ddy, dw_, x.shape, (sh, sw), pad, bf16=True).numpy()  # noqa: E731
    with split_everywhere(gpu):
        got = run()
    old = gpu.set_option("conv_split", 0)
    try:
        plain = run()
    finally:
        gpu.set_option("conv_split", old)
    for test in (np.isnan, np.isposinf, np.isneginf):
        np.testing.assert_array_equal(test(got), test(plain))
    calm = np.isfinite(plain)
    assert not calm.all() and rel_l2(got[calm], plain[calm]) <= 1e-5
    assert (got[calm] != plain[calm]).any()              # the sums of two kernels


@pytest.mark.parametrize("n,c,h,w,k,r,s,st,pad,bf16,split", [
    (32, 128, 28, 28, 256, 3, 3, 2, 1, False, True),     # strided: a compute unit for every tile
    (59, 448, 18, 18, 128, 3, 3, 2, 0, False, False),    # more tiles, few steps each
    (13, 192, 51, 51, 128, 3, 3, 2, 1, False, False),    # the second row tile half empty
    (45, 128, 32, 31, 320, 3, 3, 2, 1, False, True),     # 15000 steps and more
    (38, 256, 34, 32, 64, 3, 3, 2, 1, False, False),     # fewer than 128 filters
    (32, 128, 28, 28, 256, 3, 3, 2, 1, True, True),
    (22, 224, 54, 54, 128, 3, 3, 2, 1, True, False),     # more tiles than units, more channels than filters
    (1, 512, 32, 32, 352, 2, 2, 2, 0, True, False),      # one tap a class
    (1, 512, 7, 7, 512, 3, 3, 1, 1, True, True),
    (14, 23, 48, 48, 32, 4, 2, 1, 0, True, False),       # 32 channels to at most 32 rows
    (53, 10, 12, 87, 64, 4, 1, 1, 0, True, False),       # ... and few products for them: 256,
    (45, 7, 22, 80, 96, 4, 1, 1, 0, True, False),        # 384 in 155 tiles,
    (2, 13, 99, 199, 96, 4, 1, 1, 0, True, False),       # in two images of a tile,
    (28, 18, 39, 157, 64, 4, 1, 1, 0, True, False),      # also in more tiles than units,
    (32, 37, 12, 156, 128, 2, 2, 1, 1, True, False),     # and for more rows,
    (11, 6, 30, 30, 64, 3, 2, 1, 1, True, True),         # in one, 20 tiles
    (3, 9, 12, 11, 32, 3, 3, 2, 1, True, False),         # 32 channels to at most 32 rows, strided
    (6, 65, 10, 10, 32, 7, 7, 2, 3, True, True),         # more rows
    (1, 83, 7, 7, 32, 7, 7, 2, 3, True, False),          # ... of few pixels
    (3, 9, 12, 11, 64, 3, 3, 2, 1, True, True),          # more channels
    (44, 160, 47, 45, 64, 2, 2, 1, 1, True, False),      # more tiles than units: four taps an image,
    (40, 64, 54, 54, 64, 3, 3, 1, 1, True, True),        # nine,
    (20, 128, 64, 64, 64, 3, 3, 1, 0, True, False),      # six and three
])
def test_which_kernel_a_data_gradient_takes(gpu, n, c, h, w, k, r, s, st, pad, bf16, split):
    """By the rule on either side of its lines: the split kernel's sums have another order than the others'."""
    K = gpu.kernels
    _, wt, _, dy, _ = _data(n, c, h, w, k, r, s, st, st, pad, gpu)
    dw_, ddy = gpu.to_device(wt), gpu.to_device(dy)
    run = lambda: K.conv2d_bwd_data(ddy, dw_, (n, c, h, w), (st, st), pad, bf16=bf16).numpy()  # noqa: E731
    got = run()
    old = gpu.set_option("conv_split", 0)
    try:
        plain = run()
    finally:
        gpu.set_option("conv_split", old)
    assert rel_l2(got, plain) <= TOL
    other_bits = got.tobytes() != plain.tobytes()
    assert other_bits == split


@pytest.mark.parametrize("n,c,h,w,k,r,s,pad,split", [
    (11, 416, 54, 8, 320, 2, 2, 1, False),               # four taps over several row tiles
    (21, 384, 65, 43, 118, 2, 2, 1, True),               # ... in one
    (12, 288, 13, 51, 448, 5, 1, 0, False),              # a filter of one column: few steps,
    (14, 64, 108, 48, 480, 5, 1, 0, False),              # few of them a tile,
    (10, 448, 41, 41, 288, 1, 5, 0, True),               # 13440 steps
    (8, 192, 23, 98, 192, 3, 3, 1, False),               # three blocks of 64 rows, 7992 steps
    (45, 128, 33, 33, 192, 3, 3, 0, True),               # ... 12960
    (5, 288, 23, 59, 288, 3, 3, 0, False),               # five, 6318
    (5, 256, 46, 41, 320, 3, 3, 1, True),                # ... 8208
    (32, 128, 28, 28, 256, 3, 3, 1, True),
])
def test_which_kernel_a_strided_forward_takes(gpu, n, c, h, w, k, r, s, pad, split):
    """By the rule on either side of its lines, as above."""
    K = gpu.kernels
    x, wt, b, _, _ = _data(n, c, h, w, k, r, s, 2, 2, pad, gpu)
    dx, dw, db = gpu.to_device(x), gpu.to_device(wt), gpu.to_device(b)
    got = K.conv2d_fwd(dx, dw, db, (2, 2), pad).numpy()
    old = gpu.set_option("conv_split", 0)
    try:
        plain = K.conv2d_fwd(dx, dw, db, (2, 2), pad).numpy()
    finally:
        gpu.set_option("conv_split", old)
    assert rel_l2(got, plain) <= TOL
    assert (got.tobytes() != plain.tobytes()) == split


@pytest.mark.parametrize("count", [1, 20, 21, 43])
def test_layouts_made_in_one_call(gpu, count):
    """A launch takes the layouts of 20 filters: bit-identical to the layout that a call makes for itself, also where a filter
    of another size has a launch of its own in between."""
    import ctypes
    from xshinnosuke_amd.backend import capi
    K = gpu.kernels
    geometries = [(2, 17, 9, 9, 65, 3, 3, 1, 1, 1), (1, 40, 12, 11, 64, 3, 3, 2, 2, 1), (1, 20, 8, 8, 18, 5, 5, 1, 1, 2),
                  (1, 130, 7, 7, 24, 3, 3, 1, 1, 1)]
    calls, jobs = [], (capi.PackJob * count)()
    with split_everywhere(gpu):
        for i in range(count):
            dims, pass_ = geometries[i % 4], (i // 4) % 2
            n, c, h, w, k, r, s, sh, sw, pad = dims
            rng = np.random.default_rng(i)
            wt = gpu.to_device(he_normal(rng, (k, c, r, s)))
            oh, ow = K.conv_out_hw(h, w, r, s, (sh, sw), pad)
            x = gpu.to_device(rng.standard_normal((n, k, oh, ow) if pass_ else (n, c, h, w)).astype(np.float32))
            ref = (K.conv2d_bwd_data(x, wt, (n, c, h, w), (sh, sw), pad) if pass_ else K.conv2d_fwd(x, wt, None, (sh, sw), pad)).numpy()
            size = capi.lib.raw("xsmi_conv2d_pass_workspace_bytes")(*dims, pass_, 0)
            ws = gpu.empty(((size + 3) // 4,))
            jobs[i].w, jobs[i].workspace, jobs[i].workspace_bytes = wt.ptr, ws.ptr, size
            for field, v in zip(("N", "C", "H", "W", "K", "R", "S", "sh", "sw", "pad", "pass_"), dims + (pass_,)):
                setattr(jobs[i], field, v)
            calls.append((dims, pass_, wt, x, ws, size, ref))
        capi.lib.call("xsmi_conv2d_pack", count, ctypes.cast(jobs, ctypes.c_void_p))
        capi.lib.call("xsmi_conv2d_bwd_join")
        for i, (dims, pass_, wt, x, ws, size, ref) in enumerate(calls):
            assert jobs[i].packed == 1
            y = gpu.empty(ref.shape)
            if pass_:
                capi.lib.call("xsmi_conv2d_bwd_data", x.ptr, wt.ptr, y.ptr, *dims, 0.0, capi.CONV_WS_PACKED, ws.ptr, size)
            else:
                capi.lib.call("xsmi_conv2d_fwd", x.ptr, wt.ptr, None, y.ptr, None, *dims, capi.CONV_WS_PACKED, ws.ptr, size)
            assert y.numpy().tobytes() == ref.tobytes()


def test_weight_gradient_of_values_that_do_not_split(gpu):
    K = gpu.kernels
    x, wt, b, dy, _ = _data(2, 20, 12, 13, 70, 3, 3, 1, 1, 1, gpu)
    x[0, 3, 2, 2], x[0, 5, 8, 9], x[1, 19, 6, 6] = np.inf, np.nan, np.float32(3.4e38)
    dy[1, 4, 5, 5] = -np.inf
    _, col = oracle.conv2d_fwd(x, wt, b, (1, 1), 1)
    with np.errstate(all="ignore"):
        _, ref, _ = oracle.conv2d_bwd(dy, x.shape, wt, col, (1, 1), 1, np.zeros_like(x), np.zeros_like(wt), np.zeros_like(b))
    with split_everywhere(gpu):
        gw, _ = K.conv2d_bwd_weight(gpu.to_device(dy), gpu.to_device(x), wt.shape, (1, 1), 1, want_db=True)
    got = gw.numpy()
    for test in (np.isnan, np.isposinf, np.isneginf):
        np.testing.assert_array_equal(test(got), test(ref))
    calm = np.isfinite(ref) & (np.abs(ref) < 1e30)
    assert calm.any() and rel_l2(got[calm], ref[calm]) <= TOL


@pytest.mark.parametrize("w,pad", [(13, 1), (16, 1), (7, 1), (32, 1), (16, 0)])      # rows that end with a stage and inside one
@pytest.mark.parametrize("column", [0, -1])
@pytest.mark.parametrize("value", [np.nan, np.inf])
def test_weight_gradient_of_a_border_column_that_is_not_finite(gpu, w, pad, column, value):
    """Under some taps a border column of dy meets only padding: zero times such a value is NaN, as in the reference's
    product over the padded matrix."""
    x, wt, b, dy, _ = _data(2, 70, 9, w, 66, 3, 3, 1, 1, pad, gpu)
    dy[1, 65, 4, column] = value
    dy[0, 3, 0, column] = -value
    _, col = oracle.conv2d_fwd(x, wt, b, (1, 1), pad)
    with np.errstate(all="ignore"):
        _, ref, db_ref = oracle.conv2d_bwd(dy, x.shape, wt, col, (1, 1), pad, np.zeros_like(x), np.zeros_like(wt), np.zeros_like(b))
    with split_everywhere(gpu):
        gw, gb = gpu.kernels.conv2d_bwd_weight(gpu.to_device(dy), gpu.to_device(x), wt.shape, (1, 1), pad, want_db=True)
    for got, want in ((gw.numpy(), ref), (gb.numpy(), db_ref)):
        for test in (np.isnan, np.isposinf, np.isneginf):
            np.testing.assert_array_equal(test(got), test(want))
        calm = np.isfinite(want)
        assert calm.any() and rel_l2(got[calm], want[calm]) <= TOL


@pytest.mark.parametrize("w,column", [(w, c) for w in (16, 17, 18, 32, 40) for c in (0, 15, 16, -1) if c < w])
def test_weight_gradient_formed_again_by_some_workgroups_only(gpu, w, column):
    """One value that is not finite: the workgroups that meet it form all their sums again, the others do not, and together
    they have every product once."""
    x, wt, b, dy, _ = _data(6, 40, 9, w, 66, 3, 3, 1, 1, 1, gpu)
    x[0, 31, 5, column] = np.nan
    dy[3, 60, 4, column] = np.inf
    _, col = oracle.conv2d_fwd(x, wt, b, (1, 1), 1)
    with np.errstate(all="ignore"):
        _, ref, _ = oracle.conv2d_bwd(dy, x.shape, wt, col, (1, 1), 1, np.zeros_like(x), np.zeros_like(wt), np.zeros_like(b))
    with split_everywhere(gpu):
        got = gpu.kernels.conv2d_bwd_weight(gpu.to_device(dy), gpu.to_device(x), wt.shape, (1, 1), 1)[0].numpy()
    for test in (np.isnan, np.isposinf, np.isneginf):
        np.testing.assert_array_equal(test(got), test(ref))
    calm = np.isfinite(ref)
    assert calm.any() and rel_l2(got[calm], ref[calm]) <= TOL


def test_values_that_do_not_split_are_multiplied_one_by_one(gpu):
    """Infinities, NaN and floats that round to a bf16 infinity: the outputs they touch are the float32 ones, signs and
    NaNs included, and no other output is disturbed."""
    K = gpu.kernels
    x, wt, b, _, _ = _data(2, 20, 12, 13, 70, 3, 3, 1, 1, 1, gpu)
    clean, _ = oracle.conv2d_fwd(x, wt, b, (1, 1), 1)
    x[0, 3, 2, 2], x[0, 5, 8, 9], x[1, 19, 6, 6], x[1, 0, 0, 12] = np.inf, -np.inf, np.nan, np.float32(3.4e38)
    with np.errstate(all="ignore"):
        ref, _ = oracle.conv2d_fwd(x, wt, b, (1, 1), 1)
    with split_everywhere(gpu):
        y = K.conv2d_fwd(gpu.to_device(x), gpu.to_device(wt), gpu.to_device(b), (1, 1), 1).numpy()
    for test in (np.isnan, np.isposinf, np.isneginf):
        np.testing.assert_array_equal(test(y), test(ref))
    calm = np.isfinite(ref) & (ref == clean)
    assert calm.sum() > 0.7 * calm.size and rel_l2(y[calm], ref[calm]) <= TOL
    large = np.isfinite(ref) & ~calm                       # 3.4e38 times a weight: one term decides
    assert large.any() and np.abs(y[large] / ref[large] - 1).max() <= 1e-6


@pytest.mark.parametrize("scale", [2.0 ** -104, 2.0 ** -116, 2.0 ** -122])
def test_small_values_keep_their_last_bits(gpu, scale):
    """Below 2^-110 a value's third piece is lost: the results are formed from the products instead.  Powers of two are exact,
    so the bound is that of ordinary values."""
    K = gpu.kernels
    x, wt, b, dy, _ = _data(2, 20, 12, 13, 70, 3, 3, 1, 1, 1, gpu)
    y_ref, col = oracle.conv2d_fwd(x, wt, 0 * b, (1, 1), 1)
    dx_ref, dw_ref, _ = oracle.conv2d_bwd(dy, x.shape, wt, col, (1, 1), 1, np.zeros_like(x), np.zeros_like(wt), np.zeros_like(b))
    up = 1.0 / scale
    small = lambda a: gpu.to_device(a * np.float32(scale))  # noqa: E731
    dx_, dw_ = gpu.to_device(x), gpu.to_device(wt)
    with split_everywhere(gpu):
        y = K.conv2d_fwd(small(x), dw_, None, (1, 1), 1).numpy()
        gx = K.conv2d_bwd_data(small(dy), dw_, x.shape, (1, 1), 1).numpy()
        gw, _ = K.conv2d_bwd_weight(small(dy), dx_, wt.shape, (1, 1), 1, want_db=True)
    for got, ref in ((y, y_ref), (gx, dx_ref), (gw.numpy(), dw_ref)):
        assert rel_l2(got.astype(np.float64) * up, ref) <= TOL


@pytest.mark.parametrize("which", ["activations", "filter"])
@pytest.mark.parametrize("small,large", [(-116, 40), (-124, 100), (-130, 60), (-140, 110), (-148, 120)])
def test_small_values_against_large_ones(gpu, which, small, large):
    """Values below 2^-110, subnormal ones among them, whose products are ordinary again: the bound is that of ordinary values,
    of what is left of them as float32."""
    K = gpu.kernels
    x, wt, b, dy, _ = _data(2, 20, 12, 13, 70, 3, 3, 1, 1, 1, gpu)
    down, up = np.float32(2.0 ** small), np.float32(2.0 ** large)
    rest = 2.0 ** -(small + large)
    xs_, ws_ = (x * down, wt * up) if which == "activations" else (x * up, wt * down)
    ds = dy * (down if which == "activations" else up)
    dw = dy * (up if which == "activations" else down)               # against the input of the weight gradient
    wide = lambda a, e: np.ldexp(a.astype(np.float64), -e).astype(np.float32)  # noqa: E731 -- what float32 kept, scaled back
    e1, e2 = (small, large) if which == "activations" else (large, small)
    y_ref, col = oracle.conv2d_fwd(wide(xs_, e1), wide(ws_, e2), 0 * b, (1, 1), 1)
    dx_ref, _, _ = oracle.conv2d_bwd(wide(ds, e1), x.shape, wide(ws_, e2), col, (1, 1), 1, np.zeros_like(x), np.zeros_like(wt), np.zeros_like(b))
    _, dw_ref, _ = oracle.conv2d_bwd(wide(dw, e2), x.shape, wt, col, (1, 1), 1, np.zeros_like(x), np.zeros_like(wt), np.zeros_like(b))
    with split_everywhere(gpu):
        y = K.conv2d_fwd(gpu.to_device(xs_), gpu.to_device(ws_), None, (1, 1), 1).numpy()
        gx = K.conv2d_bwd_data(gpu.to_device(ds), gpu.to_device(ws_), x.shape, (1, 1), 1).numpy()
        gw, _ = K.conv2d_bwd_weight(gpu.to_device(dw), gpu.to_device(xs_), wt.shape, (1, 1), 1, want_db=True)
    for got, ref in ((y, y_ref), (gx, dx_ref), (gw.numpy(), dw_ref)):
        assert rel_l2(got.astype(np.float64) * rest, ref) <= TOL


@pytest.mark.parametrize("value", [2.0 ** -111, 2.0 ** -149])
def test_one_small_value_is_found_wherever_it_lies(gpu, value):
    """One value below 2^-110 and zeros around it, so that the results are its products alone: at the first and last places
    of octets, slots, rows and tiles."""
    K = gpu.kernels
    n, c, h, w, k = 2, 40, 9, 18, 66
    _, wt, _, _, _ = _data(n, c, h, w, k, 3, 3, 1, 1, 1, gpu)
    wt *= np.float32(2.0 ** 60)
    places = [(0, 0, 0, 0), (0, 7, 0, 17), (1, 8, 8, 0), (1, 39, 8, 17), (0, 15, 4, 7), (1, 16, 3, 8), (0, 31, 5, 15), (1, 32, 2, 16)]
    rest = np.float64(1.0 / value) * 2.0 ** -60
    with split_everywhere(gpu):
        for i, q in enumerate(places):
            x, dy = np.zeros((n, c, h, w), np.float32), np.zeros((n, k, h, w), np.float32)
            x[q] = value
            xr = np.zeros_like(x); xr[q] = 1
            y_ref, col = oracle.conv2d_fwd(xr, (wt * np.float32(2.0 ** -60)), None, (1, 1), 1)
            y = K.conv2d_fwd(gpu.to_device(x), gpu.to_device(wt), None, (1, 1), 1).numpy()
            assert rel_l2(y.astype(np.float64) * rest, y_ref) <= TOL, q
            # the weight gradient, once with the small value in the input and once in dy
            big = np.random.default_rng(i).standard_normal(dy.shape).astype(np.float32)
            _, ref, _ = oracle.conv2d_bwd(big, x.shape, wt, col, (1, 1), 1, np.zeros_like(x), np.zeros_like(wt), np.zeros(k, np.float32))
            gw = K.conv2d_bwd_weight(gpu.to_device(big * np.float32(2.0 ** 60)), gpu.to_device(x), wt.shape, (1, 1), 1)[0].numpy()
            assert rel_l2(gw.astype(np.float64) * rest, ref) <= TOL, q
            dy[(q[0], q[1] + 26) + q[2:]] = value
            dr = (dy / np.float32(value)).astype(np.float32) if value > 2.0 ** -120 else (dy > 0).astype(np.float32)
            big = np.random.default_rng(i).standard_normal(x.shape).astype(np.float32)
            _, col = oracle.conv2d_fwd(big, wt, None, (1, 1), 1)
            _, ref, _ = oracle.conv2d_bwd(dr, x.shape, wt, col, (1, 1), 1, np.zeros_like(x), np.zeros_like(wt), np.zeros(k, np.float32))
            gw = K.conv2d_bwd_weight(gpu.to_device(dy), gpu.to_device(big * np.float32(2.0 ** 60)), wt.shape, (1, 1), 1)[0].numpy()
            assert rel_l2(gw.astype(np.float64) * rest, ref) <= TOL, q


def test_a_partial_tile_that_never_comes_is_reported(gpu):
    K = gpu.kernels
    x, wt, b, _, _ = _data(1, 512, 7, 7, 512, 3, 3, 1, 1, 1, gpu)
    ref, _ = oracle.conv2d_fwd(x, wt, b, (1, 1), 1)
    args = [gpu.to_device(a) for a in (x, wt, b)]
    out = gpu.empty(ref.shape)
    gpu.synchronize()
    old = gpu.set_option("sk_spin_limit", 0)
    try:
        K.conv2d_fwd(*args, (1, 1), 1, out=out)
        with pytest.raises(gpu.XsmiError, match="gave up waiting"):
            gpu.synchronize()
    finally:
        gpu.set_option("sk_spin_limit", old)
    for _ in range(2):
        assert rel_l2(K.conv2d_fwd(*args, (1, 1), 1, out=out).numpy(), ref) <= TOL


@pytest.mark.parametrize("n,c,h,w,k,r,s,stride,pad", [
    (2, 48, 14, 19, 70, 3, 3, 1, 1),         # neither channel count has a bf16 kernel
    (1, 33, 9, 31, 90, 7, 7, 2, 3),
    (2, 16, 20, 11, 18, 5, 5, 1, 0),         # the fewest channels that the split kernels take
    (2, 2, 28, 37, 40, 7, 7, 2, 3),          # forward in bf16, backward-data from 40 channels
])
def test_bf16_calls_without_a_bf16_kernel_have_float32_precision(gpu, n, c, h, w, k, r, s, stride, pad):
    K = gpu.kernels
    x, wt, b, dy, _ = _data(n, c, h, w, k, r, s, stride, stride, pad, gpu)
    y_ref, col = oracle.conv2d_fwd(x, wt, b, (stride, stride), pad)
    dx_ref, _, _ = oracle.conv2d_bwd(dy, x.shape, wt, col, (stride, stride), pad, np.zeros_like(x), np.zeros_like(wt), np.zeros_like(b))
    dx_, dw_, db_, ddy = (gpu.to_device(a) for a in (x, wt, b, dy))
    if c > 8:
        mask = gpu.empty(y_ref.shape, np.uint8)
        y = K.conv2d_fwd(dx_, dw_, db_, (stride, stride), pad, relu=True, neg_mask=mask, bf16=True).numpy()
        assert rel_l2(y, np.maximum(y_ref, 0)) <= TOL
    dx = K.conv2d_bwd_data(ddy, dw_, x.shape, (stride, stride), pad, bf16=True).numpy()
    assert rel_l2(dx, dx_ref) <= TOL


@pytest.mark.parametrize("n,c,h,w,k,r,stride,pad,most", [
    (32, 128, 28, 28, 256, 3, 2, 1, 2.5),    # strided tiles of 128 x 128: measured 1.3 (before the sums that have settled: 4.5)
    (32, 64, 56, 56, 64, 3, 1, 1, 3.0),      # the even deal: 1.8 (4.7)
    (32, 3, 224, 224, 64, 7, 2, 3, 3.0),     # a first layer: 1.5 (5.2)
    (1, 512, 7, 7, 512, 3, 1, 1, 2.5),       # tiles with workgroups of their own: 1.8 (3.0)
])
def test_nan_throughout_costs_its_first_terms(gpu, n, c, h, w, k, r, stride, pad, most):
    """A sum that has become a NaN is not followed to its end; sums beside it, finite and infinite, are."""
    K = gpu.kernels
    rng = np.random.default_rng(k + h)
    x, wt = rng.standard_normal((n, c, h, w)).astype(np.float32), he_normal(rng, (k, c, r, r))
    dw = gpu.to_device(wt)

    def forward(host):
        dx, best = gpu.to_device(host), np.inf
        y = K.conv2d_fwd(dx, dw, None, (stride, stride), pad).numpy()
        gpu.profiling(True)
        try:
            for _ in range(12):
                K.conv2d_fwd(dx, dw, None, (stride, stride), pad)
                best = min(best, gpu.last_kernel_ms())
        finally:
            gpu.profiling(False)
        return y, best

    y, ordinary = forward(x)
    none, slow = forward(np.full_like(x, np.nan))
    assert np.isnan(none).all()
    assert slow <= most * ordinary, (slow, ordinary)
    mixed = x.copy()
    mixed[0, 0] = np.nan                               # settles with the first channel ...
    mixed[-1, c - 1, h - 1, :3] = np.inf               # ... does not until the last one, in the same tile where n = 1
    got, _ = forward(mixed)
    plain = _plain(gpu, mixed, dw, stride, pad)
    for test in (np.isnan, np.isposinf, np.isneginf):
        np.testing.assert_array_equal(test(got), test(plain))
    same = np.isfinite(got[1:])
    np.testing.assert_array_equal(got[1:][same], y[1:][same])


def _plain(gpu, x, dw, stride, pad):
    """The same on the fp32 matrix instructions."""
    old = gpu.set_option("conv_split", 0)
    try:
        return gpu.kernels.conv2d_fwd(gpu.to_device(x), dw, None, (stride, stride), pad).numpy()
    finally:
        gpu.set_option("conv_split", old)
