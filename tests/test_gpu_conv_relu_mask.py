"""A convolution with the ReLU in its own epilogue: the signs that it keeps for the backward are those of the fp32 matrix
instructions' sums, also where another kernel would be the fastest, and everything behind them follows from that mask."""
import ctypes

import numpy as np
import pytest

import oracle
import xshinnosuke_amd as xs
from util import he_normal, rel_l2
from xshinnosuke_amd.backend import capi
from xshinnosuke_amd.nn import functional as F

pytestmark = pytest.mark.gpu

LAYERS = [   # n c h w k r pad: geometries that the split-operand kernel serves when no mask is kept
    (2, 24, 45, 61, 40, 5, 2),
    (2, 64, 28, 28, 64, 3, 1),
    (1, 40, 16, 16, 130, 3, 1),
    (3, 16, 9, 7, 20, 2, 0),
]


def _layer(n, c, h, w, k, r, pad):
    rng = np.random.default_rng(n + c + k + h)
    x = rng.standard_normal((n, c, h, w)).astype(np.float32)
    wt, b = he_normal(rng, (k, c, r, r)), (0.1 * rng.standard_normal((1, k))).astype(np.float32)
    dy = rng.standard_normal((n, k, h + 2 * pad - r + 1, w + 2 * pad - r + 1)).astype(np.float32)
    return x, wt, b, dy


@pytest.mark.parametrize("n,c,h,w,k,r,pad", LAYERS)
def test_the_mask_is_the_fp32_kernels_and_the_gradients_follow_it(gpu, n, c, h, w, k, r, pad):
    x, wt, b, dy = _layer(n, c, h, w, k, r, pad)
    device = lambda a: xs.Tensor(gpu.to_device(a), requires_grad=True)  # noqa: E731
    tx, tw, tb = device(x), device(wt), device(b)
    out = []
    for _ in range(2):                                   # the second forward finds the filter's layout in place
        for t in (tx, tw, tb):
            t.zero_grad()
        y = F.conv2d(tx, tw, tb, (1, 1), pad, activation="relu")
        act, mask = y.eval.numpy(), y.cache["neg_mask"].numpy()
        y.backward(xs.Tensor(gpu.to_device(dy)))
        out.append((act, mask, tx.grad.eval.numpy(), tw.grad.eval.numpy(), tb.grad.eval.numpy()))
    for first, second in zip(*out):
        assert first.tobytes() == second.tobytes()
    act, mask, gx, gw, gb = out[0]
    old = gpu.set_option("conv_split", 0)                # the fp32 kernels whatever the geometry
    try:
        ref_mask = gpu.empty(act.shape, np.uint8)
        ref = gpu.kernels.conv2d_fwd(*(gpu.to_device(a) for a in (x, wt, b.reshape(-1))), (1, 1), pad, relu=True, neg_mask=ref_mask)
        assert act.tobytes() == ref.numpy().tobytes() and mask.tobytes() == ref_mask.numpy().tobytes()
    finally:
        gpu.set_option("conv_split", old)
    # the gradients of this very mask: a sign within rounding of zero is a decision, everything else is arithmetic
    y_ref, col = oracle.conv2d_fwd(x, wt, b.reshape(-1), (1, 1), pad)
    assert rel_l2(act, np.where(mask, 0, y_ref)) <= 1e-6
    refs = oracle.conv2d_bwd(np.where(mask, 0, dy).astype(np.float32), x.shape, wt, col, (1, 1), pad, np.zeros_like(x),
                             np.zeros_like(wt), np.zeros(k, np.float32))
    for got, want in zip((gx, gw, gb.reshape(-1)), refs):
        assert rel_l2(got, want) <= 1e-6                 # sums of at most 5,490 float32 products, as in the split kernels' tests


@pytest.mark.parametrize("n,c,h,w,k,r,pad", LAYERS)
def test_a_layout_made_ahead_is_the_one_the_call_reads(gpu, n, c, h, w, k, r, pad):
    """xsmi_conv2d_pack's pass 3 and XSMI_CONV_FP32_PIPE pick the same kernel, in a workspace of pass 3's own size and in one
    with room for every kernel."""
    x, wt, b, _ = _layer(n, c, h, w, k, r, pad)
    dims = (n, c, h, w, k, r, r, 1, 1, pad)
    dx, dw = gpu.to_device(x), gpu.to_device(wt)
    ref = gpu.kernels.conv2d_fwd(dx, dw, None, (1, 1), pad, fp32_pipe=True)
    for size in (capi.lib.raw("xsmi_conv2d_pass_workspace_bytes")(*dims, 0, capi.CONV_FP32_PIPE), capi.lib.raw("xsmi_conv2d_workspace_bytes")(*dims)):
        ws, y = gpu.empty(((size + 3) // 4,)), gpu.empty(ref.shape)
        job = (capi.PackJob * 1)()
        job[0].w, job[0].workspace, job[0].workspace_bytes = dw.ptr, ws.ptr, size
        for field, v in zip(("N", "C", "H", "W", "K", "R", "S", "sh", "sw", "pad", "pass_"), dims + (3,)):
            setattr(job[0], field, v)
        capi.lib.call("xsmi_conv2d_pack", 1, ctypes.cast(job, ctypes.c_void_p))
        capi.lib.call("xsmi_conv2d_bwd_join")
        flags = capi.CONV_FP32_PIPE | (capi.CONV_WS_PACKED if job[0].packed else 0)
        capi.lib.call("xsmi_conv2d_fwd", dx.ptr, dw.ptr, None, y.ptr, None, *dims, flags, ws.ptr, size)
        assert y.numpy().tobytes() == ref.numpy().tobytes()
