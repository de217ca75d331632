"""Forward and weight gradient of few products a result (csrc/conv_thin.hip) against the oracle."""
import numpy as np
import pytest

import oracle
from test_gpu_conv_variants import options
from util import he_normal

pytestmark = pytest.mark.gpu

# n c h w k r s sh sw pad: every width of the gathered row (4, 8, 16, 32 products) at its edges, filters around the groups of 2, 4,
# 8 and 32, pixels around 256 and 512 and over several images, borders wider than the image's inside, strides, one pixel; then many
# filters, which leave few splits of the weight gradient: 2 to 8 pixels a thread, the last split ragged, for 4, 8, 16 and 32 products
GEOMETRIES = [
    (1, 1, 1, 1, 1, 1, 1, 1, 1, 0), (2, 1, 28, 28, 8, 2, 2, 1, 1, 0), (3, 4, 16, 32, 9, 1, 1, 1, 1, 0), (7, 1, 19, 27, 33, 2, 2, 1, 2, 1),
    (2, 5, 16, 16, 7, 1, 1, 1, 1, 0), (3, 2, 13, 11, 32, 2, 2, 2, 1, 2), (5, 1, 12, 9, 31, 3, 3, 1, 1, 1), (2, 8, 17, 15, 130, 1, 1, 1, 1, 0),
    (4, 1, 9, 40, 5, 1, 11, 1, 2, 5), (2, 16, 8, 33, 6, 1, 1, 1, 1, 0), (1, 1, 23, 23, 3, 4, 4, 3, 3, 3), (2, 17, 9, 9, 3, 1, 1, 1, 1, 0),
    (3, 3, 14, 18, 65, 3, 3, 1, 1, 1), (2, 1, 12, 12, 2, 5, 5, 2, 2, 4), (2, 32, 7, 11, 5, 1, 1, 1, 1, 0), (300, 1, 21, 20, 4, 2, 2, 1, 1, 0),
    (9, 1, 41, 40, 301, 2, 2, 1, 1, 0), (9, 2, 30, 31, 300, 2, 2, 1, 1, 0), (12, 1, 33, 35, 257, 4, 4, 1, 1, 1), (5, 3, 40, 41, 130, 3, 3, 1, 1, 0),
]


@pytest.mark.parametrize("geom", GEOMETRIES)
def test_few_products_against_the_oracle(gpu, geom):
    n, c, h, w, k, r, s, sh, sw, pad = geom
    K = gpu.kernels
    rng = np.random.default_rng(sum(geom))
    x = rng.standard_normal((n, c, h, w)).astype(np.float32)
    wt = he_normal(rng, (k, c, r, s))
    b = rng.standard_normal((k,)).astype(np.float32)
    oh, ow = K.conv_out_hw(h, w, r, s, (sh, sw), pad)
    dy = rng.standard_normal((n, k, oh, ow)).astype(np.float32)
    y_ref, col = oracle.conv2d_fwd(x, wt, b, (sh, sw), pad)
    dw0 = rng.standard_normal(wt.shape).astype(np.float32); db0 = rng.standard_normal((k,)).astype(np.float32)
    _, dw_ref, db_ref = oracle.conv2d_bwd(dy, x.shape, wt, col, (sh, sw), pad, np.zeros_like(x), dw0.copy(), db0.copy())
    _, dw_abs, db_abs = oracle.conv2d_bwd(np.abs(dy), x.shape, wt, np.abs(col), (sh, sw), pad, np.zeros_like(x), np.abs(dw0), np.abs(db0))
    y_abs, _ = oracle.conv2d_fwd(np.abs(x), np.abs(wt), np.abs(b), (sh, sw), pad)
    dx_, dw_, db_, ddy = (gpu.to_device(a) for a in (x, wt, b, dy))
    u = 2.0 ** -24
    with options(gpu, conv_thin=2, conv_split=0):
        y = K.conv2d_fwd(dx_, dw_, db_, (sh, sw), pad).numpy()
        assert (np.abs(y - y_ref) <= (c * r * s + 3) * u * y_abs).all()      # one chain of products, the bias, the oracle's rounding
        mask = gpu.empty(y.shape, np.uint8)
        act = K.conv2d_fwd(dx_, dw_, db_, (sh, sw), pad, relu=True, neg_mask=mask).numpy()
        np.testing.assert_array_equal(act, np.maximum(y, 0.0))
        np.testing.assert_array_equal(mask.numpy(), (y < 0).astype(np.uint8))
        gw, gb = gpu.to_device(dw0), gpu.to_device(db0)
        K.conv2d_bwd_weight(ddy, dx_, wt.shape, (sh, sw), pad, dw=gw, db=gb, accumulate=True)
        # pixels of a thread (the last geometries are planned with 2 to 8; a small workspace halves the splits), 6 + 2 sums over the wave
        # and the workgroup, two roundings of the result
        bound = (16 if k >= 130 and n * h * w > 8000 else 1) + 10
        assert (np.abs(gw.numpy() - dw_ref) <= bound * u * dw_abs).all()
        assert (np.abs(gb.numpy() - db_ref) <= 3 * u * db_abs).all()
        only, _ = K.conv2d_bwd_weight(ddy, dx_, wt.shape, (sh, sw), pad)
    assert (np.abs(only.numpy() + dw0.astype(np.float64) - dw_ref) <= bound * u * dw_abs).all()


def test_groups_of_filters_in_a_large_forward(gpu):
    """536 workgroups of pixels, each with the filters in groups of 32: two groups, the second of eight."""
    K = gpu.kernels
    rng = np.random.default_rng(5)
    x, wt, b = rng.standard_normal((67, 1, 63, 63)).astype(np.float32), he_normal(rng, (40, 1, 2, 2)), rng.standard_normal((40,)).astype(np.float32)
    y_ref, _ = oracle.conv2d_fwd(x, wt, b, (1, 1), 1)
    y_abs, _ = oracle.conv2d_fwd(np.abs(x), np.abs(wt), np.abs(b), (1, 1), 1)
    y = K.conv2d_fwd(gpu.to_device(x), gpu.to_device(wt), gpu.to_device(b), (1, 1), 1).numpy()
    assert (np.abs(y - y_ref) <= 7 * 2.0 ** -24 * y_abs).all()


@pytest.mark.parametrize("n,c,h,w,k,r,s,stride,thin", [
    (45, 16, 190, 26, 74, 1, 1, 2, False),       # strided, 16 products: 4.1e6 results
    (9, 16, 190, 26, 74, 1, 1, 2, True),         # 0.8e6
    (45, 16, 190, 26, 32, 1, 1, 2, True),        # one group of filters
    (37, 11, 70, 70, 125, 1, 1, 1, False),       # stride 1, 1 x 1: 2.3e7
    (20, 11, 70, 70, 125, 1, 1, 1, True),
    (170, 1, 44, 16, 440, 3, 3, 1, False),       # stride 1, 3 x 3: 4.4e7
    (70, 1, 44, 16, 440, 3, 3, 1, True),
])
def test_large_forwards_of_many_filters_go_to_the_generic_kernel(gpu, n, c, h, w, k, r, s, stride, thin):
    """It was up to 2.8 times as fast there.  The sums' order tells the kernels apart."""
    K = gpu.kernels
    rng = np.random.default_rng(k)
    x, wt = gpu.to_device(rng.standard_normal((n, c, h, w)).astype(np.float32)), gpu.to_device(he_normal(rng, (k, c, r, s)))
    b = gpu.to_device(rng.standard_normal((k,)).astype(np.float32))
    got = K.conv2d_fwd(x, wt, b, (stride, stride), 0).numpy()
    with options(gpu, conv_thin=0):
        generic = K.conv2d_fwd(x, wt, b, (stride, stride), 0).numpy()
    with options(gpu, conv_thin=2):
        every = K.conv2d_fwd(x, wt, b, (stride, stride), 0).numpy()
    assert (generic != every).any()
    np.testing.assert_array_equal(got, every if thin else generic)


def test_a_large_strided_forward_of_six_products(gpu):
    """Too few products for the order to show: the time does (measured 36 us and, by the vector units, 57)."""
    K = gpu.kernels
    rng = np.random.default_rng(6)
    x, wt = gpu.to_device(rng.standard_normal((354, 6, 50, 50)).astype(np.float32)), gpu.to_device(he_normal(rng, (122, 6, 1, 1)))

    def best(mode):
        with options(gpu, conv_thin=mode):
            gpu.profiling(True)
            try:
                times = []
                for _ in range(12):
                    K.conv2d_fwd(x, wt, None, (2, 2), 0)
                    times.append(gpu.last_kernel_ms())
            finally:
                gpu.profiling(False)
        return min(times)

    generic, every, rule = best(0), best(2), best(1)
    assert rule < (generic + every) / 2 < every, (generic, every, rule)


@pytest.mark.parametrize("geom", [(196, 5, 26, 26, 14, 1, 3, 2, 2, 0), (98, 16, 18, 18, 1, 1, 1, 1, 1, 0), (32, 1, 17, 17, 5, 3, 3, 1, 1, 1),
                                  (33, 1, 17, 17, 5, 2, 2, 1, 1, 0)])
def test_weight_gradient_of_some_thirty_to_a_hundred_splits(gpu, geom):
    """120, 124, 37 and 33 splits: their sums were a chain of loads (16 us for the first two, 9 now, the table-driven kernel 14)."""
    n, c, h, w, k, r, s, sh, sw, pad = geom
    K = gpu.kernels
    rng = np.random.default_rng(k + r)
    x, wt = rng.standard_normal((n, c, h, w)).astype(np.float32), he_normal(rng, (k, c, r, s))
    oh, ow = K.conv_out_hw(h, w, r, s, (sh, sw), pad)
    dy = rng.standard_normal((n, k, oh, ow)).astype(np.float32)
    _, col = oracle.conv2d_fwd(x, wt, np.zeros(k, np.float32), (sh, sw), pad)
    zero = np.zeros_like(x)
    _, dw_ref, db_ref = oracle.conv2d_bwd(dy, x.shape, wt, col, (sh, sw), pad, zero, np.zeros_like(wt), np.zeros(k, np.float32))
    _, dw_abs, db_abs = oracle.conv2d_bwd(np.abs(dy), x.shape, wt, np.abs(col), (sh, sw), pad, zero, np.zeros_like(wt), np.zeros(k, np.float32))
    dx_, ddy = gpu.to_device(x), gpu.to_device(dy)
    dw, db = gpu.empty(wt.shape), gpu.empty((k,))
    K.conv2d_bwd_weight(ddy, dx_, wt.shape, (sh, sw), pad, dw=dw, db=db)
    u = 2.0 ** -24
    assert (np.abs(dw.numpy() - dw_ref) <= 11 * u * dw_abs).all()      # one pixel a thread; 6 + 2 sums, two roundings
    assert (np.abs(db.numpy() - db_ref) <= 3 * u * db_abs).all()

    def best(mode):
        with options(gpu, conv_thin=mode):
            times = []
            for _ in range(6):
                events = [gpu.Event() for _ in range(2)]
                events[0].record()
                for _ in range(10):
                    K.conv2d_bwd_weight(ddy, dx_, wt.shape, (sh, sw), pad, dw=dw, db=db)
                events[1].record()
                times.append(events[0].elapsed_ms(events[1]))
        return min(times)

    assert best(1) < best(0)
