// Convolution with very few products a result (C*R*S up to 32): forward, and weight and bias gradient.
//
//     y[n][k][m]  = bias[k] + sum over j of w[k][j] * x[n][at(m, j)]           j = (c*R + r)*S + s
//     dw[k][j]   += sum over (n, m) of dy[n][k][m] * x[n][at(m, j)]            db[k] += sum over (n, m) of dy[n][k][m]
//
// Neither is a matrix product worth its tiles: the 64-row tiles of the generic kernels multiply zeros in 15 of 16 places (4 products,
// 8 filters), and both passes are bound by reading x and dy and writing y once.  So a thread owns pixels, holds the J values
// of x under the filter in registers and uses them for a group of filters.  The forward keeps the filters in the LDS
// (every lane reads the same 16 bytes); the weight gradient keeps a group's KB x J sums in registers, adds them over the wave by
// halving (a lane hands half of its sums to its partner at each step: V + log steps instead of V log), over the
// waves through the LDS, and over the workgroups in a second launch, in float64.
// Against the generic kernels, whole operations (launch by launch, of which about 7 and 11 us are the host's):
//     256 x 1 x 28 x 28 -> 8, 2 x 2          forward 13.3 -> 8.4 us    weight gradient 34 -> 12.6
//     1024 x 1 x 28 x 28 -> 8, 2 x 2                 34 -> 8                            96 -> 15
//     32 x 8 x 56 x 56 -> 128, 1 x 1                 20 -> 13                           37 -> 25
//     32 x 1 x 112 x 112 -> 256, 2 x 2              136 -> 100 (3.9 TB/s)              222 -> 123
// Error against 64 bits: forward the same, weight gradient 0.3 to 0.5 of before, bias gradient 0.3 to 0.6.
#include "xsmi_internal.h"

namespace {

constexpr int MAX_J = 32;

struct ThinParams {
    const float *x, *w, *bias, *dy;
    float *y;
    uint8_t *mask;
    float *part, *dbpart;      // [splits][K][J], [splits][K]
    uint32_t x_bytes;
    int K, J, H, W, CHW, OHW, OW, sh, sw;
    int M;                     // pixels of all images
    int pixels;                // of a split (weight gradient)
    int relu;
    xsmi::FastDiv dOHW, dOW;
    int off[MAX_J];            // of position j from the pixel's corner, in elements
    short dr[MAX_J], ds[MAX_J];
};

// The J values of x under the filter at pixel m (zero outside the image), and where the pixel's results start.
template <int JP>
__device__ __forceinline__ void thin_gather(float (&xv)[JP], const ThinParams &p, __amdgpu_buffer_rsrc_t xr, int m, uint32_t &n, int &pix) {
    n = xsmi::fdiv((uint32_t)m, p.dOHW);
    pix = m - (int)n * p.OHW;
    const int oh = (int)xsmi::fdiv((uint32_t)pix, p.dOW), ow = pix - oh * p.OW;
    const int ihb = oh * p.sh, iwb = ow * p.sw, base = (int)n * p.CHW + ihb * p.W + iwb;
#pragma unroll
    for (int j = 0; j < JP; ++j) {
        const bool ok = j < p.J && (unsigned)(ihb + p.dr[j]) < (unsigned)p.H && (unsigned)(iwb + p.ds[j]) < (unsigned)p.W;
        const uint32_t off = ok ? (uint32_t)(base + p.off[j]) * 4u : 0xffffffffu;
        xv[j] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(xr, (int)off, 0, 0));
    }
}

// A thread: two pixels 256 apart, KT filters of blockIdx.y's group.
template <int JP, int KT>
__global__ void __launch_bounds__(256) thin_fwd_kernel(ThinParams p) {
    __shared__ __attribute__((aligned(16))) float ws[KT][JP];
    __shared__ float bs[KT];
    const int t = threadIdx.x, k0 = blockIdx.y * KT, kn = min(KT, p.K - k0);
    for (int i = t; i < KT * JP; i += 256) {
        const int k = i / JP, j = i % JP;
        ws[k][j] = k < kn && j < p.J ? p.w[(size_t)(k0 + k) * p.J + j] : 0.f;
    }
    if (t < KT) bs[t] = p.bias && t < kn ? p.bias[k0 + t] : 0.f;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void *)p.x, 0, (int)p.x_bytes, 0x00020000);
    float xv[2][JP];
    size_t at[2];
    bool live[2];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        const int m = blockIdx.x * 512 + a * 256 + t;
        uint32_t n;
        int pix;
        live[a] = m < p.M;
        thin_gather<JP>(xv[a], p, xr, live[a] ? m : 0, n, pix);
        at[a] = ((size_t)n * p.K + k0) * p.OHW + pix;
    }
    __syncthreads();
    for (int k = 0; k < kn; ++k) {
        float acc[2] = {0.f, 0.f};
#pragma unroll
        for (int j = 0; j < JP; ++j)
#pragma unroll
            for (int a = 0; a < 2; ++a) acc[a] = fmaf(ws[k][j], xv[a][j], acc[a]);
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            float v = acc[a] + bs[k];
            if (!live[a]) continue;
            const size_t o = at[a] + (size_t)k * p.OHW;
            if (p.relu) {
                if (p.mask) p.mask[o] = v < 0.f ? 1 : 0;
                v = v > 0.f ? v : 0.f;
            }
            p.y[o] = v;
        }
    }
}

// Sums of V values (a power of two up to 64) over the 64 lanes of a wave: lane l ends with the sum of value l % V in v[0].
template <int V, int N = V, int D = 32, typename T>
__device__ __forceinline__ void wave_sums(T (&v)[V], int lane) {
    if constexpr (D >= 1) {
        constexpr int M = N > D ? N / 2 : N;                   // each lane keeps the half that its bit names, or all
        const bool hi = (lane & D) != 0;
#pragma unroll
        for (int i = 0; i < M; ++i) {
            if constexpr (N > D) {
                const T keep = hi ? v[i + M] : v[i], send = hi ? v[i] : v[i + M];
                v[i] = keep + __shfl_xor(send, D);
            } else {
                v[i] += __shfl_xor(v[i], D);
            }
        }
        wave_sums<V, M, D / 2>(v, lane);
    }
}

// Split blockIdx.x of the pixels, filters KB * blockIdx.y on.  KB * JP is 64 or less.
template <int JP, int KB>
__global__ void __launch_bounds__(256) thin_wgrad_kernel(ThinParams p) {
    constexpr int V = JP * KB;
    __shared__ float red[4][V];
    __shared__ double dred[4][KB];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, k0 = blockIdx.y * KB;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void *)p.x, 0, (int)p.x_bytes, 0x00020000);
    float acc[V];
    double dbs[KB];            // the bias gradient has no products to bound its precision: its sums of up to M values are kept in 64 bits
#pragma unroll
    for (int i = 0; i < V; ++i) acc[i] = 0.f;
#pragma unroll
    for (int k = 0; k < KB; ++k) dbs[k] = 0.;
    const int m1 = min(p.M, ((int)blockIdx.x + 1) * p.pixels);
    for (int m = blockIdx.x * p.pixels + t; m < m1; m += 256) {
        float xv[JP], g[KB];
        uint32_t n;
        int pix;
        thin_gather<JP>(xv, p, xr, m, n, pix);
        const float *dy = p.dy + ((size_t)n * p.K + k0) * p.OHW + pix;
#pragma unroll
        for (int k = 0; k < KB; ++k) g[k] = k0 + k < p.K ? dy[(size_t)k * p.OHW] : 0.f;
#pragma unroll
        for (int k = 0; k < KB; ++k) {
            dbs[k] += (double)g[k];
#pragma unroll
            for (int j = 0; j < JP; ++j) acc[k * JP + j] = fmaf(g[k], xv[j], acc[k * JP + j]);
        }
    }
    wave_sums<V>(acc, lane);
    wave_sums<KB>(dbs, lane);
    if (lane < V) red[wave][lane] = acc[0];
    if (lane < KB) dred[wave][lane] = dbs[0];
    __syncthreads();
    if (t < V) {
        const int k = k0 + t / JP, j = t % JP;
        if (k < p.K && j < p.J)
            p.part[((size_t)blockIdx.x * p.K + k) * p.J + j] = (red[0][t] + red[1][t]) + (red[2][t] + red[3][t]);
    } else if (p.dbpart && t < V + KB && k0 + t - V < p.K) {
        const int k = t - V;
        p.dbpart[(size_t)blockIdx.x * p.K + k0 + k] = (float)((dred[0][k] + dred[1][k]) + (dred[2][k] + dred[3][k]));
    }
}

ThinParams thin_params(const float *x, int N, int C, int H, int W, int K, int R, int S, int sh, int sw, int pad, int OH, int OW) {
    ThinParams p = {};
    p.x = x;
    p.x_bytes = (uint32_t)((size_t)N * C * H * W * 4);
    p.K = K; p.J = C * R * S; p.H = H; p.W = W; p.CHW = C * H * W; p.OHW = OH * OW; p.OW = OW; p.sh = sh; p.sw = sw;
    p.M = N * OH * OW;
    p.dOHW = xsmi::make_fastdiv(p.OHW); p.dOW = xsmi::make_fastdiv(OW);
    for (int j = 0; j < p.J; ++j) {
        const int c = j / (R * S), r = j / S % R - pad, s = j % S - pad;
        p.off[j] = (c * H + r) * W + s;
        p.dr[j] = (short)r; p.ds[j] = (short)s;
    }
    return p;
}

template <int JP, int KB>
void launch_thin_wgrad(const ThinParams &p, int splits) {
    hipLaunchKernelGGL((thin_wgrad_kernel<JP, KB>), dim3(splits, xsmi::ceil_div(p.K, KB)), dim3(256), 0, xsmi::stream(), p);
}
template <int JP>
void launch_thin_fwd(const ThinParams &p) {
    // filters for a thread: all of a group's filters share its x; few groups while the pixels alone fill the chip
    const int blocks = xsmi::ceil_div(p.M, 512);
    if (blocks >= 2 * xsmi::cu_count() || p.K <= 8)
        hipLaunchKernelGGL((thin_fwd_kernel<JP, 32>), dim3(blocks, xsmi::ceil_div(p.K, 32)), dim3(256), 0, xsmi::stream(), p);
    else
        hipLaunchKernelGGL((thin_fwd_kernel<JP, 8>), dim3(blocks, xsmi::ceil_div(p.K, 8)), dim3(256), 0, xsmi::stream(), p);
}

}  // namespace

namespace xsmi {

// Up to 16 products the forward is the faster one up to 32 filters, which share a gather of x, and in launches that the generic kernel does
// not fill; of 1350 layers it takes 0.71 of the time (18 to 32 products: only while it is small, 27 products, 3 MB 10.8 -> 8.5; 27 MB
// 17 -> 20).  It gathers x again for every 32 (8) filters, though, and reads half of every line under a stride, while the generic
// kernel's tile is free of zeros from 64 filters on.  Not, therefore (generic -> this one, us),
//   strided, 9 products and more: from 3e6 results on (45 x 16 x 190 x 26 -> 74, 1 x 1 / 2: 14.0 -> 23.8; 285 x 15 x 50 x 50 -> 248: 62 -> 175;
//     139 x 3 x 27 x 27 -> 316, 2 x 2 / 2, 8.6e6 results: 18.5 -> 16.9; 58 x 58 -> 120, 1 x 3 / 2, 1.6e7: 25 -> 31; below 0.72 in the mean);
//   strided, 5 to 8 products for more than 96 filters: from 2.5e7 results on (354 x 6 x 50 x 50 -> 122, 1 x 1 / 2: 36 -> 57; at 2.2e7 0.95);
//   stride 1, 9 products and more for more than 96 filters: from 1.4e7 results on at 1 x 1 (37 x 11 x 70 x 70 -> 125: 30 -> 36), where
//     neighbouring taps share no lines, from 2e7 on otherwise (169 x 1 x 44 x 16 -> 440, 3 x 3: 47 -> 50; 147 x 2 x 56 x 10 -> 416, 1 x 5,
//     2.1e7: 26 -> 29; 56 x 3 x 42 x 42 -> 184, 2 x 2, 1.9e7: 27 -> 25).
bool thin_fwd_ok(int C, int K, int R, int S, int sh, int sw, int pad, long pixels) {
    const long mode = option(OPT_CONV_THIN);
    const int J = C * R * S;
    if (!mode || pad >= 32768 || J > (mode == 2 ? MAX_J : 16)) return false;
    if (mode == 2 || K <= 32) return true;
    const double results = (double)pixels * K;
    if (sh > 1 || sw > 1) return J > 8 ? results < 3e6 : J <= 4 || K <= 96 || results < 2.5e7;
    return J <= 8 || K <= 96 || results < (R * S == 1 ? 1.4e7 : 2e7);
}

// The weight gradient gathers x again for every group of filters, while the generic kernel's tile of 64 filters is free of zeros
// from 64 on: up to 8 products always (8 products, 128 filters 37 -> 25 us), up to 16 for at most 32 filters (9 products, 32 x 112 x 112:
// 16 filters 60 -> 32, 32 filters 60 -> 45, 48 filters 60 -> 67).
bool thin_wgrad_ok(int C, int K, int R, int S, int pad) {
    const long mode = option(OPT_CONV_THIN);
    return mode && pad < 32768 && C * R * S <= (mode == 2 ? MAX_J : K <= 32 ? 16 : 8);
}

int thin_conv_fwd(const float *x, const float *w, const float *bias, float *y, uint8_t *mask, int N, int C, int H, int W, int K, int R,
                  int S, int sh, int sw, int pad, int OH, int OW, int relu) {
    ThinParams p = thin_params(x, N, C, H, W, K, R, S, sh, sw, pad, OH, OW);
    p.w = w; p.bias = bias; p.y = y; p.mask = relu ? mask : nullptr; p.relu = relu;
    prof_begin();
    if (p.J <= 4) launch_thin_fwd<4>(p);
    else if (p.J <= 8) launch_thin_fwd<8>(p);
    else if (p.J <= 16) launch_thin_fwd<16>(p);
    else launch_thin_fwd<32>(p);
    prof_end();
    XSMI_LAUNCH_CHECK("thin_fwd_kernel");
    return XSMI_OK;
}

int thin_conv_bwd_weight(const float *dy, const float *x, float *dw, float *db, int N, int C, int H, int W, int K, int R, int S, int sh,
                         int sw, int pad, int OH, int OW, int accumulate, void *workspace, size_t workspace_bytes) {
    ThinParams p = thin_params(x, N, C, H, W, K, R, S, sh, sw, pad, OH, OW);
    p.dy = dy;
    const int JP = p.J <= 4 ? 4 : p.J <= 8 ? 8 : p.J <= 16 ? 16 : 32, KB = JP == 32 ? 2 : JP == 16 ? 4 : 8;
    // Two workgroups a CU, no split below 256 pixels, and as many as the least workspace of the weight gradient holds
    const size_t split_bytes = ((size_t)K * p.J + K) * sizeof(float), room = (workspace_bytes - 512) / split_bytes;
    int splits = ceil_div(2 * cu_count(), ceil_div(K, KB));
    if (splits > ceil_div(p.M, 256)) splits = ceil_div(p.M, 256);
    if ((size_t)splits > room) splits = (int)room;
    p.pixels = (int)align_up(ceil_div(p.M, splits), 256);
    splits = ceil_div(p.M, p.pixels);
    p.part = (float *)workspace;
    float *const dbpart = (float *)((char *)workspace + align_up((size_t)splits * K * p.J * sizeof(float), 256));
    p.dbpart = db ? dbpart : nullptr;
    prof_begin();
    if (JP == 4) launch_thin_wgrad<4, 8>(p, splits);
    else if (JP == 8) launch_thin_wgrad<8, 8>(p, splits);
    else if (JP == 16) launch_thin_wgrad<16, 4>(p, splits);
    else launch_thin_wgrad<32, 2>(p, splits);
    prof_end();
    XSMI_LAUNCH_CHECK("thin_wgrad_kernel");
    return wgrad_reduce_partials(p.part, dw, dbpart, db, K, p.J, K, p.J, splits, accumulate);
}

}  // namespace xsmi
