// Forward convolution of a network's first layer (1 or 3 channels, square filters of 3, 5 or 7, stride 2) on the bf16 matrix
// pipes, operands split into three bf16 values (conv_split.hip says why the result keeps float32's precision).
//
// The reduction index is (channel, filter row, filter column s) with s padded to 8, as in conv_stem.hip: on an image row the
// eight values of output pixel x are the eight columns from 2 x on, four dwords of bf16 pairs.  An MFMA step of 16 takes two
// such runs: filter rows 2 i and 2 i + 1 of one channel, and in the end the last filter row of two channels.
//
// Work layout.  A workgroup holds the split filter of 64 output channels in the LDS (66 KB for 64 x 3 x 7 x 7) for all its
// tiles of 256 output pixels (32 x 8 or 16 x 16, whichever covers the image with fewer); eight waves of 64 channels x 32
// pixels.  The tile's input patch is fetched from the image itself (places outside it read as zero: no bordered copy), split
// once, and written to the LDS as [piece][row parity][channel][row / 2][pair of columns]; the next tile's values are in flight
// while this one multiplies, its image is the other of two.  A pixel's run starts on a dword, neighbouring pixels' a dword
// further, so the reads are of single dwords without bank conflicts: a row of 32 pixels and the same row of the other
// parity are 32 banks apart (16 pixels: two rows, 32 banks, and the other parity's 16).
//
// Bound by the matrix pipe: 256 x 3 x 224 x 224 -> 64 is 434 GFLOP of bf16 products (147 of 176 places of the reduction are
// used), 0.33 ms at the 1.3 PFLOP/s that a large library product reaches; the kernel takes 0.41, without its stores 0.34,
// without the staging 0.40; on the fp32 pipe it and its bordered copy took 0.73.  N=32: 100 -> 56 us, N=1: 15.3 -> 11.4.
// Tried and slower: an image for each wave and no barriers (0.54; the patches overlap more), the next tile's loads ahead of the
// stores (0.43), tiles of 32 x 8 for images of 112 x 112 (0.46), one form of the stores for whole and
// ragged row tiles (0.43).
#include "split3.h"

namespace {

using xsmi::bf16x8;
using xsmi::uint32x4;
using xsmi::floatx16;

constexpr int SS_THREADS = 512;

struct StemSplitParams {
    const float *in, *w, *bias;
    float *out;
    uint8_t *mask;
    uint32_t in_bytes;
    int rows, H, W, pad, OY, OX, os_n, os_k, relu;
    uint32_t tiles;                                  // of one row tile
    xsmi::FastDiv dTX, dTY;                          // tiles across, down
};

template <int R, int C, int TX>
struct StemShape {
    static constexpr int TY = 256 / TX, DW = TX + 3, ROWS = 2 * TY - 2 + R, ROWS2 = (ROWS + 1) / 2;
    static constexpr int PITCH = TX == 32 ? 36 : 32, CHANNEL = ROWS2 * PITCH;                 // dwords
    static constexpr int APART = TX == 32 ? 32 : 16;                                          // banks between the parities
    static constexpr int PARITY = (C * CHANNEL + 63 - APART) / 64 * 64 + APART, PIECE = 2 * PARITY, IMAGE = 3 * PIECE;
    static constexpr int PAIRS = R / 2, STEPS = C * PAIRS + (C + 1) / 2;
    static constexpr int ITEMS = C * ROWS * DW, TURNS = (ITEMS + SS_THREADS - 1) / SS_THREADS;
    static_assert(PARITY >= C * CHANNEL && PARITY % 64 == APART, "the parities do not overlap");
    static_assert(STEPS * 6144 + 2 * IMAGE * 4 + 256 <= 160 * 1024, "LDS");
};

// The sums of a 32 x 32 block that are not carried, formed in float64 from the image and the filter.  Rare: a wave meets it
// only where a value of its sums has no split.  8 x 3 x 224 x 224 -> 64, 7 x 7: ordinary values 22 us, NaN throughout 33, one infinity 46 (fp32
// kernel 38); N=32: 61, 92, 89 (fp32 103).  Without the test for settled sums NaN took 95 and 316; the test inside the loop over the
// terms costs 9 us.
template <int R, int C>
__device__ __forceinline__ void stem_form_again(floatx16 &r, const float *in, const float *w, uint32_t in_bytes, int rows, int H, int W,
                                                int row0, int image, int iy0, int ix0, bool mine, int lane) {
    constexpr int TERMS = C * R * R, STEPS = (TERMS + 3) / 4;
    const int l15 = lane & 15, quarter = lane >> 4;
    int iy[2], ix[2], n[2];                            // of the lane's column in either half of the block
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        iy[j] = __shfl(iy0, 16 * j + l15); ix[j] = __shfl(ix0, 16 * j + l15); n[j] = __shfl(image, 16 * j + l15);
    }
    const __amdgpu_buffer_rsrc_t rin = __builtin_amdgcn_make_buffer_rsrc((void *)in, 0, (int)in_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void *)w, 0, rows * TERMS * 4, 0x00020000);
    xsmi::FormAgain again(mine, lane);
    // a NaN throughout shows in the first terms, at the image's border after those of the padding
#pragma unroll 1
    for (int i = 0, end = 1;; end = i == 1 && STEPS > 8 ? 8 : STEPS) {
#pragma unroll 1
        for (; i < end; ++i) {
            const int k = 4 * i + quarter, c = k / (R * R), rs = k - c * (R * R), y = rs / R, s = rs - y * R;
            double a[2], b[2];
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int row = row0 + 16 * j + l15;
                const int wb = __builtin_amdgcn_raw_buffer_load_b32(rw, k < TERMS && row < rows ? (row * TERMS + k) * 4 : (int)0x80000000u, 0, 0);
                const bool there = k < TERMS && (unsigned)(iy[j] + y) < (unsigned)H && (unsigned)(ix[j] + s) < (unsigned)W;
                const uint32_t place = (uint32_t)(((n[j] * C + c) * H + iy[j] + y) * W + ix[j] + s) * 4u;
                const int xb = __builtin_amdgcn_raw_buffer_load_b32(rin, there ? (int)place : (int)0x80000000u, 0, 0);
                a[j] = (double)__builtin_bit_cast(float, wb);
                b[j] = (double)__builtin_bit_cast(float, xb);
            }
            again.add(a, b);
        }
        if (i == STEPS || again.settled()) break;
    }
    again.take(r, lane);
}

template <int R, int C, int TX>
__global__ void __launch_bounds__(SS_THREADS) stem_split_kernel(StemSplitParams p) {
    typedef StemShape<R, C, TX> S;
    __shared__ __attribute__((aligned(16))) unsigned char s_a[S::STEPS * 6144];   // [step][piece][h][64 rows][8]
    __shared__ __attribute__((aligned(16))) uint32_t s_img[2 * S::IMAGE];
    __shared__ __attribute__((aligned(16))) float s_bias[64];
    const int t = threadIdx.x, lane = t & 63, h = lane >> 5, l31 = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int tile_row0 = (int)blockIdx.y * 64;
    // an XCD's workgroups (every eighth) share a run of tiles: neighbours read each other's borders
    const uint32_t xcd = blockIdx.x & 7u, stride = gridDim.x >> 3;
    const uint32_t end = (uint32_t)(((uint64_t)(xcd + 1) * p.tiles) >> 3);
    uint32_t tile = (uint32_t)(((uint64_t)xcd * p.tiles) >> 3) + (blockIdx.x >> 3);
    if (tile >= end) return;

    const __amdgpu_buffer_rsrc_t rin = __builtin_amdgcn_make_buffer_rsrc((void *)p.in, 0, (int)p.in_bytes, 0x00020000);
    int place[S::TURNS], at[S::TURNS];               // row | column << 16; dword of the LDS image, -1: none
    int from[S::TURNS];                              // element of the image, from the patch's first on
#pragma unroll
    for (int k = 0; k < S::TURNS; ++k) {
        const int i = t + SS_THREADS * k, rr = i / S::DW, d = i - rr * S::DW, c = rr / S::ROWS, row = rr - c * S::ROWS;
        place[k] = row | (2 * d) << 16;
        at[k] = i < S::ITEMS ? (row & 1) * S::PARITY + c * S::CHANNEL + (row >> 1) * S::PITCH + d : -1;
        from[k] = (c * p.H + row) * p.W + 2 * d;
    }
    struct Place { int n, y0, x0; };
    auto tile_place = [&](uint32_t i) {
        const uint32_t q = xsmi::fdiv(i, p.dTX), n = xsmi::fdiv(q, p.dTY);
        return Place{(int)n, (int)(q - n * p.dTY.d) * S::TY, (int)(i - q * p.dTX.d) * TX};
    };
    uint32_t raw[S::TURNS][2];
    auto fetch = [&](const Place &o) {
        const int iy0 = 2 * o.y0 - p.pad, ix0 = 2 * o.x0 - p.pad;
        const int first = (o.n * C * p.H + iy0) * p.W + ix0;
#pragma unroll
        for (int k = 0; k < S::TURNS; ++k) {
            const int ix = ix0 + (place[k] >> 16);
            const bool row = at[k] >= 0 && (unsigned)(iy0 + (place[k] & 0xffff)) < (unsigned)p.H;
            const uint32_t off = (uint32_t)(first + from[k]) * 4u;
#pragma unroll
            for (int e = 0; e < 2; ++e)
                raw[k][e] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rin, row && (unsigned)(ix + e) < (unsigned)p.W ? (int)(off + 4u * e) : (int)0x80000000u, 0, 0);
        }
    };
    auto stage = [&](uint32_t *img) {
#pragma unroll
        for (int k = 0; k < S::TURNS; ++k) {
            const float a = __builtin_bit_cast(float, raw[k][0]), b = __builtin_bit_cast(float, raw[k][1]);
            xsmi::SmallTest test;
            test.add(a, b);
            uint32_t p0, p1, p2;
            xsmi::split_pair3(a, b, p0, p1, p2);
            if (at[k] >= 0) {
                img[at[k]] = test.found() ? xsmi::NAN_PAIR : p0;
                img[S::PIECE + at[k]] = p1;
                img[2 * S::PIECE + at[k]] = p2;
            }
        }
    };

    Place here = tile_place(tile);
    fetch(here);
    for (int i = t; i < S::STEPS * 128; i += SS_THREADS) {           // the filter, split
        const int step = i >> 7, hh = (i >> 6) & 1, row = tile_row0 + (i & 63);
        const bool last = step >= C * S::PAIRS;                      // the last filter row of two channels
        const int q = step - C * S::PAIRS, c = last ? 2 * q + hh : step / S::PAIRS, r = last ? R - 1 : 2 * (step - c * S::PAIRS) + hh;
        float v[8];
        xsmi::SmallTest test;
#pragma unroll
        for (int s = 0; s < 8; ++s) v[s] = s < R && row < p.rows && c < C ? p.w[((size_t)row * C + c) * (R * R) + r * R + s] : 0.f;
        uint32x4 q0, q1, q2;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            test.add(v[2 * e], v[2 * e + 1]);
            uint32_t p0, p1, p2;
            xsmi::split_pair3(v[2 * e], v[2 * e + 1], p0, p1, p2);
            q0[e] = p0; q1[e] = p1; q2[e] = p2;
        }
        if (test.found()) q0 = uint32x4{xsmi::NAN_PAIR, xsmi::NAN_PAIR, xsmi::NAN_PAIR, xsmi::NAN_PAIR};
        uint32x4 *dst = reinterpret_cast<uint32x4 *>(s_a + step * 6144) + hh * 64 + (i & 63);
        dst[0] = q0; dst[128] = q1; dst[256] = q2;
    }
    if (t < 64) s_bias[t] = p.bias && tile_row0 + t < p.rows ? p.bias[tile_row0 + t] : 0.f;
    stage(s_img);
    __syncthreads();

    const int ly = TX == 32 ? wave : 2 * wave + (l31 >> 4), lx = l31 & (TX - 1);
    const int pixel = ly * S::PITCH + lx;
    const int b_pair = pixel + h * S::PARITY, b_last = pixel + h * S::CHANNEL;
    const uint32x4 *a_lane = reinterpret_cast<const uint32x4 *>(s_a) + h * 64 + l31;
    int which = 0;
    for (;;) {
        const uint32_t next = tile + stride;
        const bool more = next < end;
        Place there = here;
        if (more) {
            there = tile_place(next);
            fetch(there);
        }
        const uint32_t *img = s_img + which * S::IMAGE;
        floatx16 large[2], small[2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) large[i][v] = small[i][v] = 0.f;
        uint32x4 a[2][2][3], b[2][3];                  // [buffer][row block][piece]
        auto read = [&](auto buf, auto step_) {
            constexpr int bf = decltype(buf)::value, step = decltype(step_)::value, q = step - C * S::PAIRS;
            const uint32_t *src = q < 0                ? img + b_pair + (step / S::PAIRS) * S::CHANNEL + (step % S::PAIRS) * S::PITCH
                                  : 2 * q + 1 < C      ? img + b_last + 2 * q * S::CHANNEL + S::PAIRS * S::PITCH
                                                       : img + pixel + 2 * q * S::CHANNEL + S::PAIRS * S::PITCH;   // both halves; the filter's second is zero
#pragma unroll
            for (int k = 0; k < 3; ++k) {
#pragma unroll
                for (int e = 0; e < 4; ++e) b[bf][k][e] = src[k * S::PIECE + e];
#pragma unroll
                for (int i = 0; i < 2; ++i) a[bf][i][k] = a_lane[step * 384 + k * 128 + 32 * i];
            }
        };
        auto multiply = [&](auto buf) {
            constexpr int bf = decltype(buf)::value;
            auto mm = [&](floatx16 &acc, const uint32x4 &x, const uint32x4 &y) {
                acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, x), __builtin_bit_cast(bf16x8, y), acc, 0, 0, 0);
            };
#pragma unroll
            for (int i = 0; i < 2; ++i) mm(small[i], a[bf][i][2], b[bf][0]);
#pragma unroll
            for (int i = 0; i < 2; ++i) mm(large[i], a[bf][i][0], b[bf][0]);
#pragma unroll
            for (int i = 0; i < 2; ++i) mm(small[i], a[bf][i][0], b[bf][2]);
#pragma unroll
            for (int i = 0; i < 2; ++i) mm(small[i], a[bf][i][1], b[bf][1]);
#pragma unroll
            for (int i = 0; i < 2; ++i) mm(small[i], a[bf][i][1], b[bf][0]);
#pragma unroll
            for (int i = 0; i < 2; ++i) mm(small[i], a[bf][i][0], b[bf][1]);
        };
        auto steps = [&](auto self, auto step_) -> void {
            constexpr int step = decltype(step_)::value;
            if constexpr (step < S::STEPS) {
                if constexpr (step + 1 < S::STEPS) read(xsmi::IC<(step + 1) & 1>{}, xsmi::IC<step + 1>{});
                multiply(xsmi::IC<step & 1>{});
                self(self, xsmi::IC<step + 1>{});
            }
        };
        read(xsmi::IC<0>{}, xsmi::IC<0>{});
        steps(steps, xsmi::IC<0>{});
        if (more) stage(s_img + (which ^ 1) * S::IMAGE);

        const int y = here.y0 + ly, x = here.x0 + lx;
        const bool mine = y < p.OY && x < p.OX;
        xsmi::CarriedTest test;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                large[i][v] += small[i][v];
                test.add(large[i][v]);
            }
        if (__builtin_amdgcn_ballot_w64(mine && !test.all()) != 0)
#pragma unroll 1
            for (int i = 0; i < 2; ++i) {
                floatx16 r = i ? large[1] : large[0];
                stem_form_again<R, C>(r, p.in, p.w, p.in_bytes, p.rows, p.H, p.W, tile_row0 + 32 * i, here.n, 2 * y - p.pad, 2 * x - p.pad, mine, lane);
                if (i) large[1] = r; else large[0] = r;
            }
        // an image's outputs from a resource of its own: a lane's offset, a row's in a scalar register
        const size_t image = (size_t)here.n * (size_t)p.os_n;
        const __amdgpu_buffer_rsrc_t rout = __builtin_amdgcn_make_buffer_rsrc((void *)(p.out + image), 0, p.os_n * 4, 0x00020000);
        const __amdgpu_buffer_rsrc_t rmask = __builtin_amdgcn_make_buffer_rsrc((void *)(p.mask + (p.mask ? image : 0)), 0, p.mask ? p.os_n : 0, 0x00020000);
        int os_k = p.os_k;
        asm("" : "+s"(os_k));                          // 64 offsets formed ahead of the loop do not fit the scalar registers
        // 0x20000000 is past every image (fewer than 2^29 outputs), four times that past its bytes; rows past the last one have
        // the last one's scalar offset, which the range check takes off the length
        const uint32_t lane_off = mine ? (uint32_t)(y * p.OX + x + 4 * h * os_k) : 0x20000000u;
        const int rows_here = p.rows - tile_row0;
        // MODE 0: bias only; 1: bias + relu; 2: bias + relu + sign mask
        auto emit = [&](auto mode, auto guard) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if (guard && 32 * i >= rows_here) break;
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const float4 bias = *reinterpret_cast<const float4 *>(&s_bias[4 * h + 32 * i + 8 * g]);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int ro = 32 * i + 8 * g + e;
                        const uint32_t row_off = (uint32_t)(tile_row0 + (!guard || ro < rows_here ? ro : rows_here - 1)) * (uint32_t)os_k;
                        const uint32_t off = !guard || ro + 4 * h < rows_here ? lane_off : 0x20000000u;
                        float v = large[i][4 * g + e] + (e == 0 ? bias.x : e == 1 ? bias.y : e == 2 ? bias.z : bias.w);
                        if (mode == 2) __builtin_amdgcn_raw_buffer_store_b8((unsigned char)(v < 0.f ? 1 : 0), rmask, (int)off, (int)row_off, 0);
                        if (mode >= 1) v = v > 0.f ? v : 0.f;
                        __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), rout, (int)(off * 4u), (int)(row_off * 4u), 0);
                    }
                }
            }
        };
        auto emit_mode = [&](auto guard) {
            if (!p.relu) emit(xsmi::IC<0>{}, guard);
            else if (!p.mask) emit(xsmi::IC<1>{}, guard);
            else emit(xsmi::IC<2>{}, guard);
        };
        if (tile_row0 + 64 <= p.rows) emit_mode(std::false_type{});
        else emit_mode(std::true_type{});
        if (!more) break;
        __syncthreads();                               // the other image is whole, this one is free
        tile = next;
        here = there;
        which ^= 1;
    }
}

// Tiles of 16 x 16 where they cover the image with fewer (112 x 112: 49 against 56); of 32 x 8, whose rows are whole cache
// lines, otherwise.
int stem_tile_width(int OY, int OX) {
    const double wide = (double)xsmi::ceil_div(OX, 32) * xsmi::ceil_div(OY, 8), square = (double)xsmi::ceil_div(OX, 16) * xsmi::ceil_div(OY, 16);
    return square < wide ? 16 : 32;
}
double stem_split_tiles(int OY, int OX) {
    const int tx = stem_tile_width(OY, OX);
    return (double)xsmi::ceil_div(OX, tx) * xsmi::ceil_div(OY, 256 / tx);
}

template <int R, int C>
void stem_split_launch(StemSplitParams p, int N, int rowtiles) {
    const int tx = stem_tile_width(p.OY, p.OX), across = xsmi::ceil_div(p.OX, tx), down = xsmi::ceil_div(p.OY, 256 / tx);
    p.tiles = (uint32_t)N * (uint32_t)(across * down);
    p.dTX = xsmi::make_fastdiv(across); p.dTY = xsmi::make_fastdiv(down);
    uint32_t groups = (uint32_t)xsmi::cu_count() & ~7u;              // one a compute unit: the filter fills half of its LDS
    const uint32_t most = (p.tiles + 7) / 8 * 8;
    if (groups > most) groups = most;
    if (groups < 8) groups = 8;
    const dim3 grid(groups, (unsigned)rowtiles);
    if (tx == 16) hipLaunchKernelGGL((stem_split_kernel<R, C, 16>), grid, dim3(SS_THREADS), 0, xsmi::stream(), p);
    else hipLaunchKernelGGL((stem_split_kernel<R, C, 32>), grid, dim3(SS_THREADS), 0, xsmi::stream(), p);
}

}  // namespace

namespace xsmi {

// Of what stem_fwd_ok serves: stride 2 in both directions, images of fewer than 2^29 outputs (byte offsets), 21 terms and
// more: with one channel and 3 x 3 or 5 x 5 taps a step of 16 has too few (8 x 1 x 112 x 112 -> 320, 5 x 5: 15.1 -> 17.0 us); and tiles
// that the image fills to five eighths, unless every tile has a compute unit.  The fp32 kernel's tiles go on from image to image, these do not
// (fp32 -> split: 244 x 1 x 12 x 12 -> 177, 7 x 7, 3 x 3 outputs in tiles of 256: 9.7 -> 17.8; 210 x 3 x 14 x 9 -> 186, 7 x 7: 16 -> 34; 89 x 3 x
// 39 x 39 -> 163, 3 x 3, 0.47 full: 20 -> 27; 77 x 1 x 56 x 21 -> 240, 0.60: 17 -> 22).  705 layers: 0.76 of the fp32 kernel's time in the mean, at
// most 1.04.
bool stem_split_pays(int N, int C, int R, int K, int sh, int sw, int OH, int OW) {
    if (option(OPT_CONV_SPLIT) == 0 || option(OPT_TAP_SK) != 1 || sh != 2 || sw != 2 || (C != 3 && R != 7) || (size_t)K * OH * OW >= ((size_t)1 << 29))
        return false;
    const double tiles = stem_split_tiles(OH, OW);
    return (double)N * tiles * ceil_div(K, 64) <= (double)cu_count() || 8.0 * OH * OW >= 5.0 * 256.0 * tiles;
}

int stem_split_fwd(const float *x, const float *w, const float *bias, float *y, uint8_t *mask, int N, int C, int H, int W, int K, int R,
                   int pad, int OH, int OW, int relu) {
    StemSplitParams p;
    p.in = x; p.w = w; p.bias = bias; p.out = y; p.mask = relu ? mask : nullptr;
    p.in_bytes = (uint32_t)((size_t)N * C * H * W * 4);
    p.rows = K; p.H = H; p.W = W; p.pad = pad; p.OY = OH; p.OX = OW; p.os_n = K * OH * OW; p.os_k = OH * OW; p.relu = relu;
    const int rowtiles = ceil_div(K, 64);
    prof_begin();
    if (C == 1) stem_split_launch<7, 1>(p, N, rowtiles);
    else if (R == 7) stem_split_launch<7, 3>(p, N, rowtiles);
    else if (R == 5) stem_split_launch<5, 3>(p, N, rowtiles);
    else stem_split_launch<3, 3>(p, N, rowtiles);
    prof_end();
    XSMI_LAUNCH_CHECK("stem_split_kernel");
    return XSMI_OK;
}

}  // namespace xsmi
