// Element-wise helpers of the conv path and the workspace query.
#include "xsmi_internal.h"

namespace xsmi {
size_t conv_fwd_ws_bytes(int C, int K, int R, int S);
size_t conv_bwd_data_ws_bytes(int C, int K, int R, int S, int sh, int sw);
size_t conv_bwd_weight_ws_bytes(int N, int C, int K, int R, int S, int OH, int OW);
}  // namespace xsmi

namespace {

// dx = (accumulate ? dx : 0) + (mask ? 0 : dy); four elements per thread when aligned.
__global__ void __launch_bounds__(256) relu_mask_bwd_kernel(const float *__restrict__ dy, const uint8_t *__restrict__ mask,
                                                             float *dx, size_t n, int accumulate) {
    size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= n) return;
    if (i + 4 <= n) {
        float4 g = *reinterpret_cast<const float4 *>(dy + i);
        uchar4 m = *reinterpret_cast<const uchar4 *>(mask + i);
        float4 o = make_float4(m.x ? 0.f : g.x, m.y ? 0.f : g.y, m.z ? 0.f : g.z, m.w ? 0.f : g.w);
        if (accumulate) {
            float4 d = *reinterpret_cast<const float4 *>(dx + i);
            o.x += d.x; o.y += d.y; o.z += d.z; o.w += d.w;
        }
        *reinterpret_cast<float4 *>(dx + i) = o;
    } else {
        for (; i < n; ++i) {
            float o = mask[i] ? 0.f : dy[i];
            if (accumulate) o += dx[i];
            dx[i] = o;
        }
    }
}

// the same masked gradient delivered to two tensors at once (both inputs of the addition in front of the ReLU)
__global__ void __launch_bounds__(256) relu_mask_bwd2_kernel(const float *__restrict__ dy, const uint8_t *__restrict__ mask,
                                                              float *dx1, float *dx2, size_t n, int acc1, int acc2) {
    size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i >= n) return;
    if (i + 4 <= n) {
        float4 g = *reinterpret_cast<const float4 *>(dy + i);
        uchar4 m = *reinterpret_cast<const uchar4 *>(mask + i);
        const float4 o = make_float4(m.x ? 0.f : g.x, m.y ? 0.f : g.y, m.z ? 0.f : g.z, m.w ? 0.f : g.w);
        float4 o1 = o, o2 = o;
        if (acc1) {
            float4 d = *reinterpret_cast<const float4 *>(dx1 + i);
            o1.x += d.x; o1.y += d.y; o1.z += d.z; o1.w += d.w;
        }
        if (acc2) {
            float4 d = *reinterpret_cast<const float4 *>(dx2 + i);
            o2.x += d.x; o2.y += d.y; o2.z += d.z; o2.w += d.w;
        }
        *reinterpret_cast<float4 *>(dx1 + i) = o1;
        *reinterpret_cast<float4 *>(dx2 + i) = o2;
    } else {
        for (; i < n; ++i) {
            const float o = mask[i] ? 0.f : dy[i];
            dx1[i] = acc1 ? dx1[i] + o : o;
            dx2[i] = acc2 ? dx2[i] + o : o;
        }
    }
}

}  // namespace

extern "C" {

size_t xsmi_conv2d_pass_workspace_bytes(int N, int C, int H, int W, int K, int R, int S, int sh, int sw, int pad, int pass,
                                        unsigned flags) {
    if (N <= 0 || C <= 0 || H <= 0 || W <= 0 || K <= 0 || R <= 0 || S <= 0 || sh <= 0 || sw <= 0 || pad < 0) return 0;
    if (H + 2 * pad < R || W + 2 * pad < S) return 0;
    const int OH = (H + 2 * pad - R) / sh + 1, OW = (W + 2 * pad - S) / sw + 1;
    // what the passes refuse; their plans below count in 32 bits
    const double lim = 536870912.0;
    if ((double)N * C * H * W >= lim || (double)N * K * OH * OW >= lim || (double)K * C * R * S >= lim) return 0;
    const bool bf16 = (flags & XSMI_CONV_BF16) != 0;
    auto larger = [](size_t a, size_t b) { return a > b ? a : b; };
    size_t m = 0;
    if (pass == 0) {
        m = xsmi::conv_fwd_ws_bytes(C, K, R, S);
        if (!bf16 && xsmi::stem_fwd_ok(N, C, H, W, K, R, S, sh, sw, pad))
            m = larger(m, xsmi::stem_fwd_ws_bytes(N, C, H, W, K, R, S, sh, sw, pad));
        // the even-split fp32 kernels read their own filter layout (their partial tiles live in the library)
        if (!bf16 && xsmi::sk_path_ok(C, K)) m = larger(m, xsmi::sk_fwd_ws_bytes(C, K, R, S));
        if (xsmi::split_may_serve(C, bf16)) m = larger(m, xsmi::split_fwd_ws_bytes(N, C, H, W, K, R, S, sh, sw, pad, OH, OW));
        // the bf16 forward takes its fastest form when the workspace also holds a channels-last copy of x
        if (bf16 && xsmi::nhwc_fwd_ok(N, C, H, W, K, R, S, pad)) m = larger(m, xsmi::nhwc_fwd_ws_bytes(N, C, H, W, K, R, S, pad));
    } else if (pass == 1) {
        m = xsmi::conv_bwd_data_ws_bytes(C, K, R, S, sh, sw);
        if (!bf16 && xsmi::sk_bwd_data_ok(C, K, R, S, sh, sw)) m = larger(m, xsmi::sk_bwd_data_ws_bytes(C, K, R, S, sh, sw));
        if (xsmi::split_may_serve(K, bf16)) m = larger(m, xsmi::split_bwd_data_ws_bytes(N, C, H, W, K, R, S, sh, sw, pad, OH, OW));
        if (bf16) m = larger(m, xsmi::split_bf16_bwd_data_ws_bytes(N, C, H, W, K, R, S, sh, sw, pad, OH, OW));
    } else if (pass == 2) {
        m = xsmi::conv_bwd_weight_ws_bytes(N, C, K, R, S, OH, OW);
        if (!bf16 && xsmi::stem_wgrad_ok(N, C, H, W, K, R, S, sh, sw, pad))
            m = larger(m, xsmi::stem_wgrad_ws_bytes(N, C, H, W, K, R, S, sh, sw, pad));
        m = larger(m, xsmi::split_wgrad_ws_bytes(N, C, H, W, K, R, S, sh, sw, pad, bf16));
    }
    return m;
}

size_t xsmi_conv2d_workspace_bytes(int N, int C, int H, int W, int K, int R, int S, int sh, int sw, int pad) {
    size_t m = 0;
    for (int pass = 0; pass < 3; ++pass)
        for (unsigned flags : {0u, (unsigned)XSMI_CONV_BF16}) {
            const size_t e = xsmi_conv2d_pass_workspace_bytes(N, C, H, W, K, R, S, sh, sw, pad, pass, flags);
            m = m > e ? m : e;
        }
    return m;
}

int xsmi_conv2d_bwd(const float *dy, const float *x, const float *w, float *dx, float *dw, float *db, int N, int C, int H,
                    int W, int K, int R, int S, int sh, int sw, int pad, float beta_dx, float beta_dw, unsigned flags,
                    void *workspace, size_t workspace_bytes, void *workspace_dw, size_t workspace_dw_bytes) {
    XSMI_REQUIRE_INIT();
    XSMI_CHECK_ARG(N > 0 && C > 0 && H > 0 && W > 0 && K > 0 && R > 0 && S > 0 && sh > 0 && sw > 0 && pad >= 0 &&
                       H + 2 * pad >= R && W + 2 * pad >= S,
                   "xsmi_conv2d_bwd: bad geometry");
    XSMI_CHECK_ARG(dy && x && w && dx && dw, "xsmi_conv2d_bwd: null tensor pointer");
    XSMI_CHECK_ARG((beta_dx == 0.f || beta_dx == 1.f) && (beta_dw == 0.f || beta_dw == 1.f), "xsmi_conv2d_bwd: beta must be 0 or 1");
    XSMI_CHECK_ARG((flags & ~(XSMI_CONV_BF16 | XSMI_CONV_DW_ASYNC | XSMI_CONV_WS_PACKED)) == 0,
                   "xsmi_conv2d_bwd: unknown flags 0x%x", flags);
    const int OH = (H + 2 * pad - R) / sh + 1, OW = (W + 2 * pad - S) / sw + 1;
    const size_t data_need = xsmi::conv_bwd_data_ws_bytes(C, K, R, S, sh, sw);
    const size_t weight_need = xsmi::conv_bwd_weight_ws_bytes(N, C, K, R, S, OH, OW);
    XSMI_CHECK_ARG(workspace && workspace_bytes >= data_need, "xsmi_conv2d_bwd: workspace of %zu bytes needed, %zu given",
                   data_need, workspace_bytes);
    XSMI_CHECK_ARG(workspace_dw && workspace_dw_bytes >= weight_need,
                   "xsmi_conv2d_bwd: weight-gradient workspace of %zu bytes needed, %zu given", weight_need, workspace_dw_bytes);
    XSMI_CHECK_ARG((char *)workspace + workspace_bytes <= (char *)workspace_dw ||
                       (char *)workspace_dw + workspace_dw_bytes <= (char *)workspace,
                   "xsmi_conv2d_bwd: the two workspaces overlap");
    const unsigned kflags = flags & XSMI_CONV_BF16;
    // The two kernels share only their inputs.  On the second stream (XSMI_CONV_DW_ASYNC: until xsmi_conv2d_bwd_join, otherwise
    // joined at once) the weight gradient runs beside what follows, but the fork and the join cost the host 18 us each, and the
    // split-operand kernels fill the chip alone.  In order on the main stream therefore, but for
    //   a data gradient by the tap-major bf16 kernel whose grid (128-pixel x 64-channel tiles) leaves compute units idle, from 4e8
    //     products on (both gradients, in order -> beside: 64 -> 192, 7 x 7 / 2 at 32 x 56, N=8: 152 -> 134 us; 256 -> 512, 3 x 3 / 2 at 14 x
    //     14, N=8: 92 -> 81; 64 -> 128, 3 x 3 / 2 at 56 x 56, N=8: 52 -> 48; 21 layers 0.79 to 1.06 of in order, 0.90 in the mean;
    //     below, 64 -> 128 at 56 x 56, N=4: 44 -> 45).  Not where more than 64 tiles have 9500 or more products for a sum of one
    //     residue class: started behind the weight gradient's workgroups, several of them land on a unit and stay there, for a time
    //     beside which the weight gradient's is short (15 -> 160, 15 x 15 / 2 at 25 x 25, N=29: 417 -> 587).  Beside the one-piece split
    //     kernel, which deals a small launch over all units, nothing is gained (512 -> 512 at 7 x 7, N=32: 101 -> 116; 128 -> 128 at 28 x
    //     28, N=8: 45 -> 58; 190 layers of up to 256 tiles 1.01 to 1.5 of in order);
    //   a data gradient of either precision with at most 48 such tiles and large filters that make 9000 or more products for a sum, a
    //     few workgroups with a long chain each, from 1e9 products on; 4e8 under the bf16 flag, whose other passes are longer.  Strided,
    //     from 25 taps on, below 7e9 products (in order -> beside, 100 -> 364, 7 x 7 / 2 at 18 x 36, N=4: 101 -> 85; 31 -> 477, 5 x 5 / 2 at
    //     19 x 19, N=16: 65 -> 63; 30 layers 0.77 to 1.00); with stride 1 from 49 taps and more than 48 channels on, below 3e9 products (98
    //     -> 160, 15 x 15 at 4 x 22, N=6: 139 -> 120; 115 -> 189, 7 x 7 at 39 x 39: 80 -> 78; 40 layers 0.87 to 1.0).  Beyond these lines
    //     the workgroups that wait for one another's parts may hold units that the weight gradient could use (116 -> 415, 5 x 5 at 20 x
    //     32, N=2: 85 -> 129; 25 -> 229, 7 x 7 at 34 x 8, N=21: 98 -> 126; 84 -> 118, 15 x 15 at 30 x 16, N=4, 4.3e9: 166 -> 184; 45 -> 435, 15 x 15
    //     at 32 x 20, N=3, 8.4e9: 296 -> 369);
    //   layers of 2e9 products or more of a sweep that goes on, in float32 too: the passes between the convolutions find room
    //     (ResNet-18 steps: 224 x 224, N=32, 3.7e9 products a layer: 3.72 -> 4.01 ms; 192 x 192, 2.7e9: 3.13 -> 3.45; 224 x 224, N=16,
    //     1.85e9: 3.00 -> 2.76; 56 x 56, N=32: 3.01 -> 2.56).  A layer by itself is faster in order (64 -> 64 at 56 x 56, N=32, 3.7e9,
    //     forward and backward: 183 -> 164; 64 -> 64 at 17 x 8, N=8: 98 -> 56).
    // Behind a weight gradient that is still on the second stream an asynchronous one goes there too, whatever its size.
    const bool async = (flags & XSMI_CONV_DW_ASYNC) != 0;
    const double products = (double)N * OH * OW * C * K * R * S;
    const long long tiles = xsmi::data_gradient_tiles(N, C, H, W);
    const bool few_tiles = kflags && products >= 4e8 && tiles <= xsmi::cu_count() &&
                           xsmi::bf16_data_gradient_by_taps(N, C, H, W, K, R, S, sh, sw, pad, OH, OW);
    const bool piles_up = few_tiles && tiles > 64 && (double)K * xsmi::ceil_div(R, sh) * xsmi::ceil_div(S, sw) >= 9500;
    const bool long_chain = tiles <= 48 && (double)K * R * S >= 9000 && products >= (kflags ? 4e8 : 1e9) &&
                            (sh * sw > 1 ? R * S >= 25 && products < 7e9 : R * S >= 49 && C > 48 && products < 3e9);
    const bool pays = few_tiles || long_chain || (async && products >= 2e9);
    const bool beside = (pays && !piles_up) || (async && xsmi::side_pending());
    int rc = beside ? xsmi::side_begin() : xsmi::side_join();    // in main-stream order: after any earlier async work
    if (rc) return rc;
    rc = xsmi_conv2d_bwd_weight(dy, x, dw, db, N, C, H, W, K, R, S, sh, sw, pad, beta_dw, kflags, workspace_dw, workspace_dw_bytes);
    if (beside) xsmi::side_end();
    if (rc == XSMI_OK)
        rc = xsmi_conv2d_bwd_data(dy, w, dx, N, C, H, W, K, R, S, sh, sw, pad, beta_dx, kflags | (flags & XSMI_CONV_WS_PACKED),
                                  workspace, workspace_bytes);
    const int rj = (beside && !async) || rc ? xsmi::side_join() : XSMI_OK;
    return rc ? rc : rj;
}

int xsmi_relu_mask_bwd(const float *dy, const uint8_t *neg_mask, float *dx, size_t n, float beta) {
    XSMI_REQUIRE_INIT();
    if (n == 0) return XSMI_OK;
    XSMI_CHECK_ARG(dy && neg_mask && dx, "xsmi_relu_mask_bwd: null pointer");
    XSMI_CHECK_ARG(beta == 0.f || beta == 1.f, "xsmi_relu_mask_bwd: beta must be 0 or 1");
    size_t threads = (n + 3) / 4;
    hipLaunchKernelGGL(relu_mask_bwd_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, xsmi::stream(), dy,
                       neg_mask, dx, n, beta == 1.f ? 1 : 0);
    XSMI_LAUNCH_CHECK("relu_mask_bwd_kernel");
    return XSMI_OK;
}

int xsmi_relu_mask_bwd2(const float *dy, const uint8_t *neg_mask, float *dx1, float beta1, float *dx2, float beta2, size_t n) {
    XSMI_REQUIRE_INIT();
    if (n == 0) return XSMI_OK;
    XSMI_CHECK_ARG(dy && neg_mask && dx1 && dx2, "xsmi_relu_mask_bwd2: null pointer");
    XSMI_CHECK_ARG(dx1 != dx2, "xsmi_relu_mask_bwd2: the two outputs must differ");
    XSMI_CHECK_ARG((beta1 == 0.f || beta1 == 1.f) && (beta2 == 0.f || beta2 == 1.f), "xsmi_relu_mask_bwd2: beta must be 0 or 1");
    XSMI_CHECK_ARG((((uintptr_t)dy | (uintptr_t)dx1 | (uintptr_t)dx2) & 15) == 0 && ((uintptr_t)neg_mask & 3) == 0,
                   "xsmi_relu_mask_bwd2: tensors must be 16-byte aligned (mask: 4)");
    size_t threads = (n + 3) / 4;
    hipLaunchKernelGGL(relu_mask_bwd2_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, xsmi::stream(), dy,
                       neg_mask, dx1, dx2, n, beta1 == 1.f ? 1 : 0, beta2 == 1.f ? 1 : 0);
    XSMI_LAUNCH_CHECK("relu_mask_bwd2_kernel");
    return XSMI_OK;
}

}  // extern "C"
