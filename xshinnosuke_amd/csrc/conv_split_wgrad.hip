// fp32 weight gradient of 3 x 3, stride-1 layers on the bf16 matrix pipes, operands split into three bf16 values as in
// conv_split.hip (six products, exact up to 2^-24 of each term).
//
//     dw[k][c][r][s] = sum over (n, y, x) of dy[n][k][y][x] * in[n][c][y + r - pad][x + s - pad]
//
// rows = 64 filters, columns = 64 channels, reduction = pixels.  An MFMA lane wants eight consecutive reduction values of
// a row in 16 bytes: eight neighbouring pixels of an image row (an octet).  The sum runs over output rows y and INPUT
// columns j, dw[r][s] = sum dy[y][j + pad - s] in[y + r - pad][j]: a filter row then moves the input by whole rows, and a
// filter column moves dy, of which there are three fragments instead of nine, by one value.  A STAGE is four octets, two
// rows of two or, for rows of at most eight pixels, four rows of one; with the rows around them it takes 8 (6) octets of
// input and 6 (8) of dy for each channel and filter, which 512 threads fetch (32 bytes contiguous each), split and write
// to the LDS as [piece][channel][octet].  All nine taps read that image.  The columns of dy in the LDS begin at pad - 2, so
// that a tap's values are the five dwords from a lane's octet on, taken 0, 1 or 2 half dwords further (v_alignbit for 1).
// Odd pitches spread the lanes of a 128-bit read (channels) over all banks; the reads a dword further are dword by dword and
// meet in a quarter of the banks (9 % of a CU's cycles at 64 -> 64, 56 x 56, N=32; one dword instead of four: no faster).
//
// Eight waves: 2 x 2 of 32 filters x 32 channels, twice; the second four take the stage's other two octets, so each wave
// multiplies one k-step of 16 pixels and nine taps (54 MFMAs) between two barriers, while its share of the next stage is
// split behind the MFMAs and the one after it is in flight.  The second half multiplies with -dy (the rows of a stage that it
// owns are split as their negatives) and is subtracted through the LDS at the end: the bf16 MFMA drops what the small
// products have below the accumulator's last bits, always downwards, and what one half loses by that the other then gains
// (24 -> 32 at 112 x 112, N=32, against 64 bits: 1.0e-6, nine tenths of it one sign, -> 4.3e-7; fp32 pipe 7.1e-7).
// Workgroups take equal runs of stages; each writes its nine 64 x 64 partial products, and one launch adds them in
// ascending order in float64.  A workgroup whose sums the split does not carry (split3.h) forms them again in float64.
#include "split3.h"

#include <string.h>

namespace {

using xsmi::bf16x8;
using xsmi::IC;
using xsmi::uint32x4;
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef double doublex4 __attribute__((ext_vector_type(4)));

constexpr int T64 = 64;
constexpr int XP = 9, YP = 9;                         // octets per channel / filter in the LDS: 8 at most, made odd
constexpr int X_PLANE = T64 * XP * 16, Y_PLANE = T64 * YP * 16;
constexpr int STAGE = 3 * (X_PLANE + Y_PLANE);
constexpr int TILE = 9 * T64 * T64;                   // floats of a workgroup's partial result
static_assert(2 * STAGE <= 9 * 16 * 256 * 4, "the stages fit where the halves are added");

struct WgParams {
    const float *dy, *x;
    float *part, *dbpart;                             // [split][k tile][c tile][tap][64][64], [split][K]
    uint32_t x_bytes, dy_bytes;
    int N, C, H, W, K, OH, OW, pad, CB, RB;           // CB octets across and RB output rows of a stage
    int kt, ct, splits, stages, per, rem;             // stages of the pass, per split
    int row_blocks, col_blocks;
};

struct Place { int n, y, x; };                        // image, first output row, first input column of a stage
__device__ __forceinline__ void next_stage(const WgParams &p, Place &q) {
    q.x += p.CB * 8;
    if (q.x >= p.col_blocks * p.CB * 8) {
        q.x = 0; q.y += p.RB;
        if (q.y >= p.row_blocks * p.RB) { q.y = 0; ++q.n; }
    }
}

// The partial result of `stages` stages from `q` on, formed from the products themselves in float64.  A workgroup decides this
// for itself, so its share is the one that it has among workgroups that do not: the stages' output rows and input columns.
// A border column of dy has no input column under some taps: it meets a zero there, as in the fp32 kernels and in the
// reference's product over the padded matrix, so that it shows if it is not finite.  Bound by the fp64 matrix pipe: a tap at a time, 16 x 16
// blocks (D: register v of lane l is row l / 16 + 4 v, column l % 16), a lane's quarter of the half's 16 pixels four deep.  All of 64 -> 64 at 56 x 56, N=8, not finite: 187 us (a product at a time behind the
// partial results: 2850).
__device__ __forceinline__ void form_again(const WgParams &p, float *part, double *s_half, Place q0, int stages, int k0, int c0,
                                        int half, int wr, int wc, int lane) {
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)p.x, 0, (int)p.x_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc((void *)p.dy, 0, (int)p.dy_bytes, 0x00020000);
    const int l15 = lane & 15, quarter = lane >> 4, octet = 2 * half + (quarter >> 1);
    const int o_row = octet / p.CB, o_col = (octet - o_row * p.CB) * 8 + (quarter & 1) * 4;
    const int row0 = wr * 32 + l15, col0 = wc * 32 + l15;
    auto at = [](__amdgpu_buffer_rsrc_t r, bool there, int index) {    // a value, zero where there is none
        const int b = __builtin_amdgcn_raw_buffer_load_b32(r, there ? (int)((uint32_t)index * 4u) : (int)0x80000000u, 0, 0);
        return (double)__builtin_bit_cast(float, b);
    };
#pragma unroll 1
    for (int tap = 0; tap < 9; ++tap) {
        const int r = tap / 3 - p.pad, s = tap % 3 - p.pad;
        doublex4 d[2][2];
#pragma unroll
        for (int i = 0; i < 4; ++i) d[i >> 1][i & 1] = doublex4{0.0, 0.0, 0.0, 0.0};
        Place q = q0;
#pragma unroll 1
        for (int st = 0; st < stages; ++st) {
            const int y = q.y + o_row, iy = y + r;
            double a[4][2], b[4][2];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int ix = q.x + o_col + i, x = ix - s;
                const bool there = y < p.OH && x >= 0 && x < p.OW, in = there && iy >= 0 && iy < p.H && ix < p.W;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int k = k0 + row0 + 16 * j, c = c0 + col0 + 16 * j;
                    a[i][j] = at(ry, there && k < p.K, ((q.n * p.K + k) * p.OH + y) * p.OW + x);
                    b[i][j] = at(rx, in && c < p.C, ((q.n * p.C + c) * p.H + iy) * p.W + ix);
                }
            }
            // columns -1 and W of the input, where the walk has no place for them
            const int beside = s < 0 && q.x == 0 ? 0 : s > 0 && q.x + p.CB * 8 == p.W ? p.OW - 1 : -1;
            if (p.pad == 1 && beside >= 0) {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const int k = k0 + row0 + 16 * j;
                    const double edge = at(ry, y < p.OH && o_col == 0 && k < p.K, ((q.n * p.K + k) * p.OH + y) * p.OW + beside);
#pragma unroll
                    for (int i = 0; i < 2; ++i) d[j][i] = __builtin_amdgcn_mfma_f64_16x16x4f64(edge, 0.0, d[j][i], 0, 0, 0);
                }
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    d[j >> 1][j & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i][j >> 1], b[i][j & 1], d[j >> 1][j & 1], 0, 0, 0);
            next_stage(p, q);
        }
        auto place = [&](int j, int v) { return (wr * 32 + 16 * (j >> 1) + quarter + 4 * v) * T64 + col0 + 16 * (j & 1); };
        if (half == 1) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) s_half[place(j, v)] = d[j >> 1][j & 1][v];
        }
        __syncthreads();
        if (half == 0) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) part[tap * T64 * T64 + place(j, v)] = (float)(d[j >> 1][j & 1][v] + s_half[place(j, v)]);
        }
        __syncthreads();
    }
}

__global__ void __launch_bounds__(512, 2) split_wgrad_kernel(WgParams p) {
    __shared__ __attribute__((aligned(16))) unsigned char s_mem[9 * 16 * 256 * 4];
    __shared__ uint32_t s_again;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int half = wave >> 2, wr = (wave >> 1) & 1, wc = wave & 1, h = lane >> 5, l31 = lane & 31;
    const int tiles = p.kt * p.ct;
    const int id = (int)xsmi::xcd_contiguous_id(blockIdx.x, gridDim.x);
    const int split = id / tiles, tile = id - split * tiles, k0 = tile / p.ct * T64, c0 = tile % p.ct * T64;
    const int s0 = split * p.per + (split < p.rem ? split : p.rem), s1 = s0 + p.per + (split < p.rem ? 1 : 0);

    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)p.x, 0, (int)p.x_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc((void *)p.dy, 0, (int)p.dy_bytes, 0x00020000);

    // ---- staging: of the stage's octets of the input this thread takes number t, and of dy, those of the first half's rows of
    // all filters first, likewise.  A thread past the last octet (8 and 6, or 6 and 8, for each of 64) stages zeros beside them.
    const int nx = (p.RB + 2) * p.CB, ny = p.RB * (p.CB + 1);          // per channel and per filter
    struct Mine { int ch, row, col, lds; bool live, own; };
    auto mine = [&](bool y) {
        Mine m;
        const int per = y ? ny / 2 : nx, part = t / (per * T64), i = t - part * per * T64, c = i / per;   // two parts of dy
        const int across = y ? p.CB + 1 : p.CB, sl = part * per + i - c * per;
        m.own = part < (y ? 2 : 1);
        m.row = sl / across; m.col = (sl - m.row * across) * 8;
        m.live = m.own && (y ? k0 + c < p.K : c0 + c < p.C);
        m.ch = y ? (k0 + c) * p.OH * p.OW : (c0 + c) * p.H * p.W;
        m.lds = y ? 3 * X_PLANE + (c * YP + (m.own ? sl : YP - 1)) * 16 : (c * XP + (m.own ? sl : XP - 1)) * 16;
        return m;
    };
    const Mine m0 = mine(false), m1 = mine(true);
    const bool minus = wave * 64 >= ny / 2 * T64;     // uniform: this wavefront's octets of dy are the second half's
    auto place = [&](int s) {
        Place q;
        const int cb = s % p.col_blocks, r = s / p.col_blocks;
        q.x = cb * p.CB * 8; q.y = r % p.row_blocks * p.RB; q.n = r / p.row_blocks;
        return q;
    };
    auto next = [&](Place &q) { next_stage(p, q); };
    float pre[2][8];
    int cut[2], early[2];                             // values from this one on are past the row; the octet begins that much early
    bool ends[2];                                     // uniform: some octet of the stage crosses an end of its row
    auto fetch = [&](auto jt, const Place &q) {
        constexpr int j = decltype(jt)::value;
        const Mine &m = j == 0 ? m0 : m1;
        constexpr bool y = j == 1;
        const int rows = y ? p.OH : p.H, cols = y ? p.OW : p.W;
        const int row = q.y + m.row - (y ? 0 : p.pad), first = q.x + (y ? p.pad - 2 : 0), col = first + m.col;
        early[j] = col < 0 ? -col : 0;                // fetched from column 0 and moved up
        cut[j] = cols - col;
        ends[j] = first < 0 || first + (p.CB + (y ? 1 : 0)) * 8 > cols;
        const int from = col < 0 ? 0 : col;
        const bool ok = m.live && row >= 0 && row < rows && from < cols;
        const uint32_t image = (uint32_t)(y ? p.K * p.OH * p.OW : p.C * p.H * p.W);
        const uint32_t off = ok ? (uint32_t)q.n * image + (uint32_t)(m.ch + row * cols + from) : 0x20000000u;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32x4 v = __builtin_amdgcn_raw_buffer_load_b128(y ? ry : rx, (int)(off * 4u) + 16 * i, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) { const uint32_t b = v[e]; pre[j][4 * i + e] = __builtin_bit_cast(float, b); }
        }
    };
    // db: the dy octets of a stage overlap by two columns on either side; the values of columns [8 i, 8 i + 8) are the ones
    // 2 - pad and further of octet i and the first of octet i + 1, so an octet adds all of its values up to a stage's end
    // and the last one the first 2 - pad only
    double db_sum = 0.0;
    const bool want_db = p.dbpart != nullptr && c0 == 0;
    uint32x4 piece[3];
    xsmi::SmallTest small;
    auto trim = [&](auto jt, const Place &q) {        // zeros outside the row; values that do not split are looked for
        constexpr int j = decltype(jt)::value;
        float *v = pre[j];
        if (ends[j]) {
#pragma unroll
            for (int n = 0; n < 2; ++n)
                if (early[j] > n) {
#pragma unroll
                    for (int i = 7; i > 0; --i) v[i] = v[i - 1];
                    v[0] = 0.f;
                }
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = i < cut[j] ? v[i] : 0.f;
        }
        small = xsmi::SmallTest{};
#pragma unroll
        for (int i = 0; i < 4; ++i) small.add(v[2 * i], v[2 * i + 1]);
        if (j == 1 && want_db) {
            const Mine &m = m1;
            const bool first = q.x == 0 || m.col > 0, last = m.col == p.CB * 8 && q.x + p.CB * 8 < p.col_blocks * p.CB * 8;
            float all = ((v[2] + v[3]) + (v[4] + v[5])) + (v[6] + v[7]);
            float head = v[0] + (p.pad == 0 ? v[1] : 0.f);
            all += p.pad == 0 ? 0.f : v[1];
            db_sum += (double)((first ? head : 0.f) + (last ? 0.f : all));
        }
    };
    auto split_two = [&](auto jt, auto it) {          // pairs 2 it and 2 it + 1
        constexpr int j = decltype(jt)::value, i0 = 2 * decltype(it)::value;
        auto two = [&](auto negative) {
#pragma unroll
            for (int i = i0; i < i0 + 2; ++i) {
                uint32_t a, b, c;
                xsmi::split_pair3<decltype(negative)::value != 0>(pre[j][2 * i], pre[j][2 * i + 1], a, b, c);
                piece[0][i] = a; piece[1][i] = b; piece[2][i] = c;
            }
        };
        if (j == 1 && minus) two(IC<1>{});
        else two(IC<0>{});
    };
    auto put = [&](auto jt, int to) {
        constexpr int j = decltype(jt)::value;
        const Mine &m = j == 0 ? m0 : m1;
        constexpr int plane = j == 1 ? Y_PLANE : X_PLANE;
        piece[0][0] = small.found() ? xsmi::NAN_PAIR : piece[0][0];    // the first dword of an octet is read under some tap
#pragma unroll
        for (int q = 0; q < 3; ++q) *reinterpret_cast<uint32x4 *>(s_mem + to + m.lds + q * plane) = piece[q];
    };

    // ---- multiply side: this lane's octet e of the stage, its filter and its channel ----
    const int e = 2 * half + h, e_row = e / p.CB, e_col = e - e_row * p.CB;
    const int a_base = 3 * X_PLANE + ((wr * 32 + l31) * YP + e_row * (p.CB + 1) + e_col) * 16;
    const int b_base = ((wc * 32 + l31) * XP + e) * 16, r_step = p.CB * 16;
    floatx16 acc[9];
#pragma unroll
    for (int i = 0; i < 9; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][v] = 0.f;
    bf16x8 fa[3][3], fb[2][3];                        // [filter column][piece], [row parity][piece]
    typedef uint32_t uint32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
    auto read_a = [&](int from) {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
            const unsigned char *src = s_mem + from + a_base + q * Y_PLANE;
            const uint32x4 d = *reinterpret_cast<const uint32x4 *>(src);
            const uint32x4 d1 = *reinterpret_cast<const uint32x4_a4 *>(src + 4);
            uint32x4 m;
#pragma unroll
            for (int i = 0; i < 4; ++i) m[i] = __builtin_amdgcn_alignbit(d1[i], d[i], 16);
            fa[2][q] = __builtin_bit_cast(bf16x8, d);
            fa[1][q] = __builtin_bit_cast(bf16x8, m);
            fa[0][q] = __builtin_bit_cast(bf16x8, d1);
        }
    };
    auto read_b = [&](auto rt, int from) {
        constexpr int r = decltype(rt)::value;
#pragma unroll
        for (int q = 0; q < 3; ++q)
            fb[r & 1][q] = *reinterpret_cast<const bf16x8 *>(s_mem + from + b_base + q * X_PLANE + r * r_step);
    };
    auto multiply = [&](auto rt, int qa, int qb) {
        constexpr int r = decltype(rt)::value;
#pragma unroll
        for (int s = 0; s < 3; ++s)
            acc[3 * r + s] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[s][qa], fb[r & 1][qb], acc[3 * r + s], 0, 0, 0);
    };

    Place at = place(s0), at1 = at;                   // of the values in flight, and of the next ones
    fetch(IC<0>{}, at); fetch(IC<1>{}, at);
    trim(IC<0>{}, at); split_two(IC<0>{}, IC<0>{}); split_two(IC<0>{}, IC<1>{}); put(IC<0>{}, 0);
    trim(IC<1>{}, at); split_two(IC<1>{}, IC<0>{}); split_two(IC<1>{}, IC<1>{}); put(IC<1>{}, 0);
    next(at);
    fetch(IC<0>{}, at); fetch(IC<1>{}, at);           // past the last image: out of range
    at1 = at;
    int cur = 0;
    for (int s = s0; s < s1; ++s) {
        xsmi::wait_lgkmcnt0();
        xsmi::block_barrier();                        // this stage is complete, and nobody reads the other one any more
        const int to = STAGE - cur;
        const bool more = s + 1 < s1;
        next(at1);
        read_b(IC<0>{}, cur);
        read_a(cur);
        read_b(IC<1>{}, cur);
        __builtin_amdgcn_sched_barrier(0);
        auto row = [&](auto rt) {
            constexpr int r = decltype(rt)::value;
            multiply(rt, 2, 0);
            if constexpr (r > 0) { if (more) trim(IC<r - 1>{}, at); }
            __builtin_amdgcn_sched_barrier(0);
            multiply(rt, 1, 0);
            if constexpr (r > 0) split_two(IC<r - 1>{}, IC<0>{});
            __builtin_amdgcn_sched_barrier(0);
            multiply(rt, 0, 0);
            if constexpr (r > 0) split_two(IC<r - 1>{}, IC<1>{});
            __builtin_amdgcn_sched_barrier(0);
            multiply(rt, 1, 1);
            if constexpr (r > 0) { if (more) put(IC<r - 1>{}, to); }
            __builtin_amdgcn_sched_barrier(0);
            multiply(rt, 0, 1);
            if constexpr (r > 0) fetch(IC<r - 1>{}, at1);
            __builtin_amdgcn_sched_barrier(0);
            multiply(rt, 0, 2);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (r == 0) read_b(IC<2>{}, cur);
        };
        row(IC<0>{});
        row(IC<1>{});
        row(IC<2>{});
        at = at1;
        cur = to;
    }

    // the two halves of the waves are added: register v of lane l is filter 8 (v / 4) + 4 (l / 32) + v % 4, channel l % 32
    // of the wave's block
    xsmi::wait_lgkmcnt0();
    __syncthreads();
    float *s_acc = reinterpret_cast<float *>(s_mem);
    if (half == 1) {
#pragma unroll
        for (int i = 0; i < 9; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) s_acc[(i * 16 + v) * 256 + (t & 255)] = acc[i][v];
    }
    if (t == 0) s_again = 0;
    __syncthreads();
    float *part = p.part + ((size_t)split * tiles + tile) * TILE;
    if (half == 0) {
        float *dst = part + (wr * 32 + 4 * h) * T64 + wc * 32 + l31;
        xsmi::CarriedTest test;
#pragma unroll
        for (int i = 0; i < 9; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const float sum = acc[i][v] - s_acc[(i * 16 + v) * 256 + t];
                test.add(sum);
                dst[i * T64 * T64 + (8 * (v >> 2) + (v & 3)) * T64] = sum;
            }
        if (!test.all()) s_again = 1;
    }
    __syncthreads();
    if (s_again) {
        xsmi::wait_vmcnt<0>();                        // what is overwritten now has been written
        __syncthreads();
        form_again(p, part, reinterpret_cast<double *>(s_mem), place(s0), s1 - s0, k0, c0, half, wr, wc, lane);
    }
    if (want_db) {                                    // a filter's octets are in up to ny threads: added in their order
        double *s_db = reinterpret_cast<double *>(s_mem);
        __syncthreads();
        if (m1.own) s_db[(m1.lds - 3 * X_PLANE) / 16] = db_sum;
        __syncthreads();
        if (t < T64 && k0 + t < p.K) {
            double sum = 0.0;
            for (int i = 0; i < ny; ++i) sum += s_db[t * YP + i];
            p.dbpart[(size_t)split * p.K + k0 + t] = (float)sum;
        }
    }
}

// dw (+)= the partial results in ascending order, in float64.  A workgroup owns 8 / GW filters and 64 channels, TAPS taps
// of them; GW waves share the splits of a filter.  Many splits (64 -> 64 channels: 256): GW = 8 and one tap, so that 576
// workgroups read the 38 MB (12.7 us; 192 of three taps: 23 us); few (512 -> 512: 4): GW = 1 and all nine taps (12.6 us;
// GW = 8: 20 us).  The workgroups behind them add db.
template <int GW, int TAPS>
__global__ void __launch_bounds__(512) split_wgrad_reduce_kernel(WgParams p, float *dw, float *db, int accumulate, int dw_blocks) {
    constexpr int KB = 8 / GW, ROW = T64 * TAPS, FLIGHT = GW == 1 ? 2 : GW == 2 ? 4 : 8;
    __shared__ double s_sum[8][ROW];
    __shared__ double s_part[512];
    const int t = threadIdx.x, c = t & 63, w = t >> 6;
    if ((int)blockIdx.x >= dw_blocks) {
        const int k = ((int)blockIdx.x - dw_blocks) * 64 + c;
        double sum = 0.0;
        if (k < p.K) {
#pragma unroll 4
            for (int s = w; s < p.splits; s += 8) sum += (double)p.dbpart[(size_t)s * p.K + k];
        }
        s_part[t] = sum;
        __syncthreads();
        if (t >= 64 || k >= p.K) return;
        sum = accumulate ? (double)db[k] : 0.0;
        for (int j = 0; j < 8; ++j) sum += s_part[j * 64 + t];
        db[k] = (float)sum;
        return;
    }
    const int r0 = (int)blockIdx.x % (9 / TAPS) * TAPS, kc = (int)blockIdx.x / (9 / TAPS), kb = kc / p.ct * KB, ctile = kc % p.ct, c0 = ctile * T64;
    const int k = kb + w / GW, tiles = p.kt * p.ct, tile = k / T64 * p.ct + ctile;
    double sum[TAPS];
#pragma unroll
    for (int i = 0; i < TAPS; ++i) sum[i] = 0.0;
    if (k < p.K) {
        const float *src = p.part + (size_t)tile * TILE + (r0 * T64 + k % T64) * T64 + c;
        const size_t step = (size_t)tiles * TILE;
        for (int s = w % GW; s < p.splits; s += GW * FLIGHT) {
            float v[FLIGHT][TAPS];
#pragma unroll
            for (int j = 0; j < FLIGHT; ++j)
#pragma unroll
                for (int i = 0; i < TAPS; ++i) v[j][i] = s + GW * j < p.splits ? src[(size_t)(s + GW * j) * step + i * T64 * T64] : 0.f;
#pragma unroll
            for (int j = 0; j < FLIGHT; ++j)
#pragma unroll
                for (int i = 0; i < TAPS; ++i) sum[i] += (double)v[j][i];
        }
    }
#pragma unroll
    for (int i = 0; i < TAPS; ++i) s_sum[w][c * TAPS + i] = sum[i];
    __syncthreads();
    const int live = (p.C - c0 < T64 ? p.C - c0 : T64) * TAPS;
    for (int o = t; o < KB * ROW; o += 512) {
        const int kk = o / ROW, i = o - kk * ROW;
        if (i >= live || kb + kk >= p.K) continue;
        float *q = dw + ((size_t)(kb + kk) * p.C + c0 + i / TAPS) * 9 + r0 + i % TAPS;
        double all = 0.0;
#pragma unroll
        for (int j = 0; j < GW; ++j) all += s_sum[kk * GW + j][i];
        *q = (float)(accumulate ? all + (double)*q : all);
    }
}

void wg_plan(WgParams &p, int N, int C, int H, int W, int K, int pad, int OH, int OW) {
    memset(&p, 0, sizeof(p));
    p.N = N; p.C = C; p.H = H; p.W = W; p.K = K; p.OH = OH; p.OW = OW; p.pad = pad;
    p.CB = W <= 8 ? 1 : 2; p.RB = 4 / p.CB;
    p.kt = xsmi::ceil_div(K, T64); p.ct = xsmi::ceil_div(C, T64);
    p.row_blocks = xsmi::ceil_div(OH, p.RB); p.col_blocks = xsmi::ceil_div(W, 8 * p.CB);
    p.stages = N * p.row_blocks * p.col_blocks;
    // splits: a stage takes about 2 us in each round of workgroups over the 256 compute units (a constant: a workspace may
    // be sized before a device is open), and a partial result 0.06 us to write and read again
    const int tiles = p.kt * p.ct;
    long best = -1;
    for (int s = 1; s <= 256 && s <= p.stages; ++s) {
        const long cost = (long)xsmi::ceil_div(tiles * s, 256) * xsmi::ceil_div(p.stages, s) * 200 + (long)tiles * s * 6;
        if (best < 0 || cost < best) { best = cost; p.splits = s; }
    }
    p.per = p.stages / p.splits; p.rem = p.stages % p.splits;
    p.x_bytes = (uint32_t)((size_t)N * C * H * W * 4); p.dy_bytes = (uint32_t)((size_t)N * K * OH * OW * 4);
}

}  // namespace

namespace xsmi {

size_t split_wgrad_ws_bytes(int N, int C, int H, int W, int K, int R, int S, int sh, int sw, int pad, bool bf16) {
    const long opt = option(OPT_CONV_SPLIT);
    if (opt == 0 || R != 3 || S != 3 || sh != 1 || sw != 1 || pad > 1) return 0;
    const int OH = H + 2 * pad - 2, OW = W + 2 * pad - 2;
    WgParams p;
    wg_plan(p, N, C, H, W, K, pad, OH, OW);
    // Below about seven stages for each compute unit the fp32 kernels' smaller partial results win (128 -> 128 at 28 x 28:
    // N=8 32 -> 38 us, N=16 45 -> 44, N=32 72 -> 60), with a few channels the columns that multiply zeros (2 -> 480 at
    // 93 x 93, N=6: 64 -> 147 us).
    if (opt < 2 && (C < 16 || (long)p.stages * p.kt * p.ct < 1750)) return 0;
    // A workgroup here fills a compute unit's LDS and registers.  A bf16 data gradient of few tiles, which is started beside the
    // weight gradient (xsmi_conv2d_bwd), then waits and lands on the first units that come free, several of its workgroups on
    // one: the fp32 kernels let it in (both gradients, 512 -> 512 at 7 x 7: N=32 235 -> 163 us, N=64 334 -> 208; 256 -> 256 at
    // 14 x 14, N=32: 117 -> 110; slower only below 100 channels, 48 -> 80 at 61 x 61, N=8: 125 -> 131).  With four times as
    // many filters as channels this kernel stays ahead (64 -> 512 at 56 x 56, N=4: 153 us, fp32 kernels 185), and so it does
    // beside a float32 data gradient (512 -> 512, N=32: 146, fp32 kernels 163) or one that fills the chip by itself (N=128: 310,
    // fp32 kernels 453).  The rule looks at the flag, so that both ways to ask for a weight gradient give the same bits.
    if (opt < 2 && bf16 && K < 4 * C && data_gradient_tiles(N, C, H, W) <= cu_count()) return 0;
    return align_up((size_t)p.splits * p.kt * p.ct * TILE * sizeof(float), 256) + align_up((size_t)p.splits * K * sizeof(float), 256);
}

int split_conv_bwd_weight(const float *dy, const float *x, float *dw, float *db, int N, int C, int H, int W, int K, int pad, int OH,
                          int OW, int accumulate, void *workspace) {
    WgParams p;
    wg_plan(p, N, C, H, W, K, pad, OH, OW);
    p.dy = dy; p.x = x;
    p.part = (float *)workspace;
    if (db) p.dbpart = (float *)((char *)workspace + align_up((size_t)p.splits * p.kt * p.ct * TILE * sizeof(float), 256));
    hipStream_t st = stream();
    prof_begin();
    hipLaunchKernelGGL(split_wgrad_kernel, dim3(p.splits * p.kt * p.ct), dim3(512), 0, st, p);
    prof_end();
    XSMI_LAUNCH_CHECK("split_wgrad_kernel");
    const int db_blocks = db ? ceil_div(K, 64) : 0;
    auto reduce = [&](auto kernel, int per_filters, int parts) {
        const int dw_blocks = ceil_div(K, per_filters) * p.ct * parts;
        hipLaunchKernelGGL(kernel, dim3(dw_blocks + db_blocks), dim3(512), 0, st, p, dw, db, accumulate, dw_blocks);
    };
    if (p.splits >= 32) reduce(split_wgrad_reduce_kernel<8, 1>, 1, 9);
    else if (p.splits >= 8) reduce(split_wgrad_reduce_kernel<2, 3>, 4, 3);
    else reduce(split_wgrad_reduce_kernel<1, 9>, 8, 1);
    XSMI_LAUNCH_CHECK("split_wgrad_reduce_kernel");
    return XSMI_OK;
}

}  // namespace xsmi
