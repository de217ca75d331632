// fp32 weight gradient on the bf16 matrix pipes, operands split into three bf16 values (six products, conv_split.hip): filters up
// to 16 x 16, any stride and padding.
//
//     dw[k][j] = sum over pixels m = (n, oy, ox) of dy[n][k][oy][ox] * in[n][c][oy sh + r - pad][ox sw + s - pad],  j = (c R + r) S + s
//
// Rows = filters, columns = j, reduction = pixels.  An OCTET is eight channels under one filter row r, and two of them are a
// SUB-IMAGE: sixteen input rows, staged once for all taps s of the filter row.  Lanes are neighbouring places of those rows
// (slots), a lane has an octet's eight values of a slot, or eight filters of a pixel of dy, as in conv_split.hip, and what it
// writes to the LDS is [piece][octet][slot][8].  The reduction index is then the one that is NOT contiguous in the LDS, and the
// fragments are read transposed (ds_read_b64_tr_b16: sixteen lanes fetch four slots of sixteen entries, and each ends up with
// the four values of its entry).  Every lane gives the place of its slot itself, so a tap, a stride and the end of a row are
// nothing but addresses, and an MFMA's 32 columns are any two UNITS (sub-image, tap).  A slot is an input column; with one tap
// across, only the columns that are read have slots.  Bank conflicts: none on large images, 1 to 6 % of a compute unit's cycles on rows
// of 7 to 14 pixels and under a stride (counted).
//
// Workgroups of eight waves: KT filters by `subs` sub-images, a stage is PX pixels.  Waves are 2 x 2 (KT = 64) or 1 x 4 (32)
// blocks of 32 rows by P pairs of units, twice: the second four take the second half of a stage's pixels, multiply with -dy and
// are subtracted at the end, which cancels what the bf16 MFMA always rounds downwards.  One image is multiplied while the next
// is split behind the MFMAs and the one after it is in flight.  Workgroups take equal runs of stages; each writes its sums as
// they lie in the registers, and one launch adds them in ascending order in float64.
//
// Kernel and reduction, before (table-driven fp32 kernel, or one for 3 x 3, stride 1 alone that took neighbouring pixels as they lie
// in memory) and now: 24 -> 40, 5 x 5 at 45 x 61, N=7: 37 -> 26 us; 32 -> 16, 7 x 7 at 109 x 109, N=5: 179 -> 53; 123 -> 296, 5 x 5
// at 50 x 27, N=3: 149 -> 63; 96 -> 16, 3 x 3 at 81 x 81, N=12: 75 -> 47.  3 x 3, stride 1, whole tiles: the kernel alone is 7 to 10 %
// slower than the one before (64 -> 64 at 56 x 56, N=32: 50.1 -> 53.8), its reduction shorter (12.6 -> 6.0), the error half (2.2e-7 ->
// 1.1e-7).  What bounds it, 123 -> 296: 55 us, the matrix pipes busy for 44 % of it, vector instructions (splitting, addresses, the
// sums) issued for 50 %, and the two hardly overlap; holding one half of the waves back or giving it priority changed nothing, a
// third image in the LDS with the barrier in the middle of the MFMAs lost 10 % (smaller stages, more addresses).
#include "split3.h"

#include <string.h>

#include <utility>

namespace {

using xsmi::bf16x8;
using xsmi::IC;
using xsmi::uint32x4;
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef double doublex4 __attribute__((ext_vector_type(4)));

constexpr int THREADS = 512;
constexpr int MAX_TAPS = 16;                          // down and across

struct WgParams {
    const float *dy, *x;
    float *part, *dbpart;                             // [split][j tile][k tile][4096 P] (as in the registers), [split][K]
    uint32_t x_bytes, dy_bytes;
    int K, C, R, S, H, W, OH, OW, OHW, in_n, plane, sh, pad, M, N, dy_next;      // dy_next: from past an image's last pixel to the next image's first
    int octets, x_last, dy_last;                      // octets of entries; last plane (row) of an octet within the buffer's bounds
    int su, sx, Wx;                                   // input columns per slot, slots per pixel and per row of pixels
    int NS, subs, units;                              // slots of an octet in the LDS, sub-images of a tile, their units
    int kt, jt, splits, stages, per, rem;
    int KT, PX, P, NJ;
    int few;                                          // sums of a few products: formed in float64
    uint32_t rOW, rOHW, rWx, rOH;                     // 2^23 over them, rounded up (small_div)
    xsmi::FastDiv dOW, dOH, dNS, dR;
};

// v / d from r = reciprocal(d), full-rate 24-bit instructions only: exact for 0 <= v <= d + SMALL_PAST, d < SMALL_DIV, as
// v r - v 2^23 / d <= v is then below 2^23 / d, and v r < 2^32.
constexpr int SMALL_DIV = 2600, SMALL_PAST = 510;
inline uint32_t reciprocal(int d) { return (1u << 23) / (uint32_t)d + 1u; }
__device__ __forceinline__ int small_div(int v, uint32_t r) { return (int)((uint32_t)__umul24((uint32_t)v, r) >> 23); }
static_assert((SMALL_DIV + SMALL_PAST) * SMALL_DIV < 1 << 23, "the error stays below one part");

template <int... I, typename F>
__device__ __forceinline__ void for_each(std::integer_sequence<int, I...>, const F &f) { (f(IC<I>{}), ...); }

struct Unit { int sub, s; };
// Unit u of a tile.  The two units of a pair are the same tap of neighbouring sub-images, which lie half the banks apart (NS = 4
// mod 8); the last sub-image of an odd number pairs its taps.
__device__ __forceinline__ Unit unit_of(const WgParams &p, int u) {
    const int paired = p.subs / 2 * 2 * p.S;
    if (u >= paired) return Unit{p.subs - 1, u - paired};
    const int i = u / (2 * p.S), rest = u - i * 2 * p.S;
    return Unit{2 * i + (rest & 1), rest >> 1};
}

struct Entry { int c, r; };
__device__ __forceinline__ Entry entry_of(const WgParams &p, int octet0, int sub, int l15) {     // channels past the last too
    const int o = octet0 + 2 * sub + (l15 >> 3), c8 = (int)xsmi::fdiv((uint32_t)o, p.dR);
    return Entry{c8 * 8 + (l15 & 7), o - c8 * p.R};
}

// The sums of a workgroup that the split does not carry (split3.h), formed from the products in float64 on the fp64 matrix
// instructions (D: register v of lane l is row l / 16 + 4 v, column l % 16): every second group of four pixels for each half of
// the waves, added through the LDS.
template <int KT, int P>
__device__ __forceinline__ void form_again(const WgParams &p, float *part, double *s_half, int m0, int m1, int k0, int octet0,
                                           int half, int wr, int wc, int lane) {
    constexpr int WC = KT == 64 ? 2 : 4;
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)p.x, 0, (int)p.x_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc((void *)p.dy, 0, (int)p.dy_bytes, 0x00020000);
    const int l15 = lane & 15, quarter = lane >> 4;
    auto at = [](__amdgpu_buffer_rsrc_t r, bool there, int index) {
        const int b = __builtin_amdgcn_raw_buffer_load_b32(r, there ? (int)((uint32_t)index * 4u) : (int)0x80000000u, 0, 0);
        return (double)__builtin_bit_cast(float, b);
    };
#pragma unroll 1
    for (int pair = 0; pair < P; ++pair) {
        int c[2], r[2], s[2];
        bool live[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int u = 2 * (wc * P + pair) + i;
            const Unit un = unit_of(p, u < p.units ? u : 0);
            const Entry en = entry_of(p, octet0, un.sub, l15);
            live[i] = u < p.units && en.c < p.C;
            c[i] = en.c; r[i] = en.r; s[i] = un.s;
        }
        doublex4 d[2][2];
#pragma unroll
        for (int i = 0; i < 4; ++i) d[i >> 1][i & 1] = doublex4{0.0, 0.0, 0.0, 0.0};
#pragma unroll 1
        for (int m4 = m0 + 4 * half; m4 < m1; m4 += 8) {
            const int m = m4 + quarter;
            const bool there = m < m1;
            const int q = (int)xsmi::fdiv((uint32_t)m, p.dOW), n = (int)xsmi::fdiv((uint32_t)q, p.dOH);
            const int ox = m - q * p.OW, oy = q - n * p.OH, pix = m - n * p.OHW;
            double a[2], b[2];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int k = k0 + wr * 32 + 16 * i + l15;
                a[i] = at(ry, there && k < p.K, (n * p.K + k) * p.OHW + pix);
                const int iy = oy * p.sh + r[i] - p.pad, ix = ox * p.sx * p.su + s[i] - p.pad;
                b[i] = at(rx, there && live[i] && iy >= 0 && iy < p.H && ix >= 0 && ix < p.W, n * p.in_n + c[i] * p.plane + iy * p.W + ix);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) d[i >> 1][i & 1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i >> 1], b[i & 1], d[i >> 1][i & 1], 0, 0, 0);
        }
        double *mine = s_half + (wr * WC + wc) * 1024 + lane;
        if (half == 1) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int v = 0; v < 4; ++v) mine[(4 * i + v) * 64] = d[i >> 1][i & 1][v];
        }
        __syncthreads();
        if (half == 0) {
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const int row = 16 * (i >> 1) + quarter + 4 * v, to = ((row >> 2) & 1) * 32 + (i & 1) * 16 + l15;
                    part[(((wr * WC + wc) * P + pair) * 4 + (row >> 3)) * 256 + to * 4 + (row & 3)] = (float)(d[i >> 1][i & 1][v] + mine[(4 * i + v) * 64]);
                }
        }
        __syncthreads();
    }
}

template <int KT, int PX, int P, int NJ>
__global__ void __launch_bounds__(THREADS, 2) split_wgrad_kernel(WgParams p) {
    constexpr int WC = KT == 64 ? 2 : 4, KS = PX / 32;
    constexpr int Y_ITEMS = KT / 8 * PX;              // (octet, pixel) of dy, then (octet, slot) of the input: one a thread and round
    constexpr int PLANE = NJ * THREADS * 16, IMAGE = 3 * PLANE;
    static_assert(Y_ITEMS <= THREADS && Y_ITEMS % 64 == 0, "dy is staged in the first round, by whole wavefronts");
    constexpr int HALF = P * 16 * 256 * 4;            // bytes of the second half's sums
    static_assert(2 * IMAGE >= THREADS * 64, "the images' LDS holds the sums of db, and a pair's of float64");
    __shared__ __attribute__((aligned(16))) unsigned char s_mem[2 * IMAGE > HALF ? 2 * IMAGE : HALF];
    __shared__ uint32_t s_again;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int half = wave >> 2, wr = KT == 64 ? (wave >> 1) & 1 : 0, wc = wave & (WC - 1);
    const int l15 = lane & 15, h = lane >> 5, odd = (lane >> 4) & 1;
    const int tiles = p.kt * p.jt;
    const int id = (int)xsmi::xcd_contiguous_id(blockIdx.x, gridDim.x);
    auto uniform = [](int v) { return __builtin_amdgcn_readfirstlane(v); };      // (the divisions leave vector registers)
    const int split = uniform(id / tiles), tile = id - split * tiles, jtile = uniform(tile / p.kt), k0 = (tile - jtile * p.kt) * KT, octet0 = jtile * p.subs * 2;
    const int s0 = split * p.per + (split < p.rem ? split : p.rem), s1 = s0 + p.per + (split < p.rem ? 1 : 0);

    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc((void *)p.x, 0, (int)p.x_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t ry = __builtin_amdgcn_make_buffer_rsrc((void *)p.dy, 0, (int)p.dy_bytes, 0x00020000);

    // ---- staging.  Values of rows and channels past the tensor's are fetched and multiplied like the others (within the buffers'
    // bounds) and dropped at the end.  Octet o of dy has its pixels four at a time at the places xor (o % 4), so that the
    // transposed reads of four octets meet in different banks.
    const bool y_wave = wave * 64 < Y_ITEMS;          // uniform: in the first round
    int slot[NJ], row[NJ];                            // pixel, or slot (< 0: none); filter row
    bool busy[NJ];                                    // uniform: the wavefront has an item in this round
    uint32_t off[NJ];                                 // bytes from an image's first value to the octet's
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int item = j * THREADS + t;
        if (j == 0 && y_wave) {
            const int o = item / PX;
            slot[j] = (item % PX) ^ (4 * (o & 3));
            row[j] = 0;
            busy[j] = true;
            off[j] = (uint32_t)(k0 + 8 * o < p.K ? k0 + 8 * o : 0) * (uint32_t)p.OHW * 4u;
        } else {
            const int xi = item - Y_ITEMS, o = (int)xsmi::fdiv((uint32_t)xi, p.dNS), at = octet0 + o;
            const bool live = o < 2 * p.subs && at < p.octets;
            const int c8 = (int)xsmi::fdiv((uint32_t)(live ? at : 0), p.dR);
            slot[j] = live ? xi - o * p.NS : -1;
            row[j] = live ? at - c8 * p.R : 0;
            busy[j] = __builtin_amdgcn_ballot_w64(o < 2 * p.subs) != 0;
            off[j] = (uint32_t)(c8 * 8 * p.plane) * 4u;
        }
    }
    const uint32_t sign = y_wave && slot[0] >= PX / 2 ? 0x80000000u : 0u;
    float pre[NJ][8];
    // What a lane does for a stage it does from the stage's first pixel on, in numbers that 24 bits hold (`small_div`).
    struct Start { int n, oy, ox, pix; };             // of the stage's first pixel (past the last: of the last)
    auto start_of = [&](int stage) {
        const int m = stage * PX < p.M ? stage * PX : p.M - 1;
        const int q = (int)xsmi::fdiv((uint32_t)m, p.dOW), n = (int)xsmi::fdiv((uint32_t)q, p.dOH);
        return Start{n, q - n * p.OH, m - q * p.OW, m - n * p.OHW};
    };
    auto place = [&](auto jt, int stage) {            // byte offset of the item's first value, past all bounds where it has none
        constexpr int j = decltype(jt)::value;
        const Start b = start_of(stage);
        uint32_t at;
        if (j == 0 && y_wave) {
            const int pix = b.pix + slot[j], n = p.OHW < PX ? small_div(pix, p.rOHW) : pix >= p.OHW ? 1 : 0;
            at = (off[j] + (uint32_t)(b.n * p.K * p.OHW + pix + n * p.dy_next) * 4u) | (slot[j] < p.M - stage * PX ? 0u : 0x80000000u);
        } else {
            const int v = b.ox * p.sx + slot[j], rows = small_div(v, p.rWx), y = b.oy + rows, n = small_div(y, p.rOH);
            const int iy = __mul24(y - __mul24(n, p.OH), p.sh) + row[j] - p.pad, ix = __mul24(v - __mul24(rows, p.Wx), p.su) - p.pad;
            const bool there = (slot[j] >= 0) & (n < p.N - b.n) & (stage * PX < p.M) & ((uint32_t)ix < (uint32_t)p.W) & ((uint32_t)iy < (uint32_t)p.H);
            at = (off[j] + (uint32_t)((b.n + n) * p.in_n + __mul24(iy, p.W) + ix) * 4u) | (there ? 0u : 0x80000000u);
        }
        return at;
    };
    auto fetch = [&](auto jt, uint32_t at) {
        constexpr int j = decltype(jt)::value;
        const bool y = j == 0 && y_wave;
        const __amdgpu_buffer_rsrc_t r = y ? ry : rx;
        const uint32_t step = (uint32_t)(y ? p.OHW : p.plane) * 4u;
        const int last = y ? p.dy_last : p.x_last;
#pragma unroll
        for (int e = 0; e < 8; ++e)
            pre[j][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)at, (int)((e <= last ? (uint32_t)e : 0u) * step), 0));
    };
    double db[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) db[e] = 0.0;
    const bool want_db = p.dbpart != nullptr && jtile == 0 && y_wave;
    uint32x4 piece[3];
    xsmi::SmallTest small;
    auto split_two = [&](auto jt, auto it) {          // pairs 2 it and 2 it + 1
        constexpr int j = decltype(jt)::value, i0 = 2 * decltype(it)::value;
        if constexpr (i0 == 0) small = xsmi::SmallTest{};
#pragma unroll
        for (int i = i0; i < i0 + 2; ++i) {
            float a = pre[j][2 * i], b = pre[j][2 * i + 1];
            if (j == 0 && want_db) { db[2 * i] += (double)a; db[2 * i + 1] += (double)b; }
            if (j == 0) {
                a = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, a) ^ sign);
                b = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, b) ^ sign);
            }
            small.add(a, b);
            uint32_t q0, q1, q2;
            xsmi::split_pair3(a, b, q0, q1, q2);
            piece[0][i] = q0; piece[1][i] = q1; piece[2][i] = q2;
        }
    };
    auto put = [&](auto jt, int to) {
        constexpr int j = decltype(jt)::value;
        unsigned char *dst = s_mem + to + (j * THREADS + t) * 16;
        const bool found = small.found();             // the octet's sums are formed again
#pragma unroll
        for (int i = 0; i < 4; ++i) piece[0][i] = found ? xsmi::NAN_PAIR : piece[0][i];
#pragma unroll
        for (int q = 0; q < 3; ++q) *reinterpret_cast<uint32x4 *>(dst + q * PLANE) = piece[q];
    };

    // ---- multiply side.  Value i of a fragment's half: pixel 16 ks + 8 h + 4 i + l15 / 4 of the half, entries 4 (l15 % 4) .. + 3
    // of its sixteen.
    const int oct = (l15 >> 1) & 1, row_oct = 2 * odd + oct, px0 = half * (PX / 2) + 8 * h + (l15 >> 2);
    int a_rd[2], b_rd[KS][2], unit_off[P];
#pragma unroll
    for (int i = 0; i < 2; ++i) a_rd[i] = ((wr * 4 + row_oct) * PX + ((px0 + 4 * i) ^ (4 * row_oct))) * 16 + (l15 & 1) * 8;
#pragma unroll
    for (int i = 0; i < P; ++i) {
        const int u = 2 * (wc * P + i) + odd;
        const Unit un = unit_of(p, u < p.units ? u : 0);
        unit_off[i] = ((2 * un.sub + oct) * p.NS + un.s) * 16;
    }
    floatx16 acc[P];
#pragma unroll
    for (int i = 0; i < P; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][v] = 0.f;
    // The MFMAs of a k-step add up from zero and the sum of a pair's is added to the accumulator in one rounding: six roundings of
    // the full sum otherwise, downwards all of them (64 -> 64 at 56 x 56, N=32: 3.7e-7 against 64 bits, 1.3e-7 this way).  Where the
    // registers hold dy's fragments of both k-steps, a pair's k-steps follow each other and are added together.
    constexpr bool BOTH = KS == 2 && P <= 4;
    constexpr int FB = P < 5 || NJ * KS < 6 ? 2 : 1;  // sets of fragments that the registers hold
    floatx16 tmp[2], zero = {};
    bf16x8 fa[BOTH ? 2 : 1][3], fb[FB][3];
    auto read = [&](int at0, int at1) {
        typedef __attribute__((address_space(3))) bf16x4 lds_x4;
        const bf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_x4 *)(s_mem + at0));
        const bf16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_x4 *)(s_mem + at1));
        return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
    };
    int cur = 0;
    auto read_a = [&](auto kt) {
        constexpr int ks = decltype(kt)::value;
#pragma unroll
        for (int q = 0; q < 3; ++q) fa[BOTH ? ks : 0][q] = read(cur + a_rd[0] + ks * 256 + q * PLANE, cur + a_rd[1] + ks * 256 + q * PLANE);
    };
    auto read_b = [&](auto it) {
        constexpr int i = decltype(it)::value, ks = BOTH ? i % KS : i / P, q0 = BOTH ? i / KS : i % P;
        const int at0 = b_rd[ks][0] + unit_off[q0], at1 = b_rd[ks][1] + unit_off[q0];
#pragma unroll
        for (int q = 0; q < 3; ++q) fb[i % FB][q] = read(at0 + q * PLANE, at1 + q * PLANE);
    };

    auto all_of = [&](auto jt, int to) { split_two(jt, IC<0>{}); split_two(jt, IC<1>{}); put(jt, to); };
    auto fetch_all = [&](int stage) {
        fetch(IC<0>{}, place(IC<0>{}, stage)); fetch(IC<1>{}, place(IC<1>{}, stage));
        if constexpr (NJ == 3) fetch(IC<NJ - 1>{}, place(IC<NJ - 1>{}, stage));
    };
    fetch_all(s0);
    all_of(IC<0>{}, 0); all_of(IC<1>{}, 0);
    if constexpr (NJ == 3) all_of(IC<NJ - 1>{}, 0);
    fetch_all(s0 + 1);
    int s = s0;
    do {                                              // at least one stage
        const int ox = start_of(s).ox;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const int px = px0 + 16 * ks + 4 * i;                 // past the last pixel: a place of the image, dy is zero there
                b_rd[ks][i] = cur + (Y_ITEMS + __mul24(px, p.sx) + __mul24(small_div(ox + px, p.rOW), p.Wx - p.OW * p.sx)) * 16 + (l15 & 1) * 8;
            }
        xsmi::wait_lgkmcnt0();
        xsmi::block_barrier();                        // this image is complete, and nobody reads the other one any more
        const int to = IMAGE - cur;
        const bool more = s + 1 < s1;
        read_a(IC<0>{});
        if constexpr (BOTH) read_a(IC<KS - 1>{});
        read_b(IC<0>{});
        __builtin_amdgcn_sched_barrier(0);
        // four operations a round, dealt over the KS P places behind three MFMAs
        auto op = [&](auto ot) {
            constexpr int o = decltype(ot)::value, j = o / 4;
            if constexpr (j < NJ) {
                if constexpr (o % 4 == 3) {
                    fetch(IC<j>{}, place(IC<j>{}, s + 2));
                }
                else if (busy[j] && more) {
                    if constexpr (o % 4 == 0) split_two(IC<j>{}, IC<0>{});
                    if constexpr (o % 4 == 1) split_two(IC<j>{}, IC<1>{});
                    if constexpr (o % 4 == 2) put(IC<j>{}, to);
                }
            }
        };
        auto add = [&](auto it) {
            constexpr int i = decltype(it)::value, q0 = BOTH ? i / KS : i % P;
            acc[q0] += tmp[(BOTH ? q0 : i) & 1];
            asm volatile("" : "+v"(acc[q0]));         // here, and not where the registers of both are needed
        };
        auto multiply = [&](auto it) {
            constexpr int i = decltype(it)::value, q0 = BOTH ? i / KS : i % P, ks = BOTH ? i % KS : i / P, b = i % FB;
            constexpr int a = BOTH ? ks : 0, T = (BOTH ? q0 : i) & 1;
            if constexpr (FB == 2 && i + 1 < KS * P) read_b(IC<i + 1>{});
            tmp[T] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[a][2], fb[b][0], BOTH && ks > 0 ? tmp[T] : zero, 0, 0, 0);
            tmp[T] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[a][1], fb[b][1], tmp[T], 0, 0, 0);
            tmp[T] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[a][0], fb[b][2], tmp[T], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (i > 0 && (!BOTH || ks == 0)) add(IC<i - 1>{});
            __builtin_amdgcn_sched_barrier(0);
            constexpr int o0 = i * 4 * NJ / (KS * P), o1 = (i + 1) * 4 * NJ / (KS * P);
            static_assert(o1 - o0 <= 6, "operations of a place");
            if constexpr (o0 + 0 < o1) op(IC<o0 + 0>{});
            if constexpr (o0 + 1 < o1) op(IC<o0 + 1>{});
            if constexpr (o0 + 2 < o1) op(IC<o0 + 2>{});
            if constexpr (o0 + 3 < o1) op(IC<o0 + 3>{});
            if constexpr (o0 + 4 < o1) op(IC<o0 + 4>{});
            if constexpr (o0 + 5 < o1) op(IC<o0 + 5>{});
            __builtin_amdgcn_sched_barrier(0);
            tmp[T] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[a][1], fb[b][0], tmp[T], 0, 0, 0);
            tmp[T] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[a][0], fb[b][1], tmp[T], 0, 0, 0);
            tmp[T] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[a][0], fb[b][0], tmp[T], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (FB == 1 && i + 1 < KS * P) read_b(IC<i + 1>{});
            if constexpr (!BOTH && q0 == P - 1 && ks + 1 < KS) read_a(IC<ks + 1>{});
        };
        for_each(std::make_integer_sequence<int, KS * P>{}, multiply);
        add(IC<KS * P - 1>{});
        cur = to;
    } while (++s < s1);

    // the halves of the waves are subtracted: register v of lane l is row 8 (v / 4) + 4 (l / 32) + v % 4 of the wave's block,
    // entry l % 16 of the pair's unit l / 16 % 2
    xsmi::wait_lgkmcnt0();
    __syncthreads();
    float *s_acc = reinterpret_cast<float *>(s_mem);
    if (half == 1) {
#pragma unroll
        for (int i = 0; i < P; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) s_acc[(i * 16 + v) * 256 + (t & 255)] = acc[i][v];
    }
    if (t == 0) s_again = 0;
    __syncthreads();
    float *part = p.part + ((size_t)split * tiles + tile) * (4096 * P);
    if (half == 0) {
        float *dst = part + (wr * WC + wc) * P * 1024 + lane * 4;
        bool again = false;
#pragma unroll
        for (int i = 0; i < P; ++i) {
            const int u = 2 * (wc * P + i) + odd;
            const bool live = u < p.units && entry_of(p, octet0, unit_of(p, u).sub, l15).c < p.C;
            xsmi::CarriedTest test;
#pragma unroll
            for (int v4 = 0; v4 < 4; ++v4) {
                float4 sum;
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    (&sum.x)[v] = acc[i][4 * v4 + v] - s_acc[(i * 16 + 4 * v4 + v) * 256 + t];
                    const bool counts = live && k0 + wr * 32 + 8 * v4 + 4 * h + v < p.K;
                    test.add(counts ? (&sum.x)[v] : 0.f);
                }
                *reinterpret_cast<float4 *>(dst + (i * 4 + v4) * 256) = sum;
            }
            again |= !test.all();
        }
        if (again) s_again = 1;
    }
    __syncthreads();
    if (s_again || p.few) {
        xsmi::wait_vmcnt<0>();                        // what is overwritten now has been written
        __syncthreads();
        const int m1 = s1 * PX < p.M ? s1 * PX : p.M;
        form_again<KT, P>(p, part, reinterpret_cast<double *>(s_mem), s0 * PX, m1, k0, octet0, half, wr, wc, lane);
    }
    if (p.dbpart != nullptr && jtile == 0) {          // a filter's pixels are in PX threads: added in their order
        double *s_db = reinterpret_cast<double *>(s_mem);
        __syncthreads();
        if (y_wave) {
#pragma unroll
            for (int e = 0; e < 8; ++e) s_db[(t / PX * 8 + e) * PX + slot[0]] = db[e];
        }
        __syncthreads();
        if (t < KT && k0 + t < p.K) {
            double sum = 0.0;
            for (int i = 0; i < PX; ++i) sum += s_db[t * PX + ((i + t) & (PX - 1))];
            p.dbpart[(size_t)split * p.K + k0 + t] = (float)sum;
        }
    }
}

// dw (+)= the partial results in ascending order, in float64.  A workgroup owns 256 sums that lie together in a partial result
// (a kilobyte for each of G waves, which share the splits); the workgroups behind them add db.
template <int G>
__global__ void __launch_bounds__(64 * G) split_wgrad_reduce_kernel(WgParams p, float *dw, float *dbias, int accumulate, int dw_blocks) {
    constexpr int FLIGHT = 4;
    __shared__ double s_sum[G][4][64];
    const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
    double sum[4] = {0.0, 0.0, 0.0, 0.0};
    if ((int)blockIdx.x >= dw_blocks) {
        const int k = ((int)blockIdx.x - dw_blocks) * 64 + lane;
        if (k < p.K) {
#pragma unroll 4
            for (int s = g; s < p.splits; s += G) sum[0] += (double)p.dbpart[(size_t)s * p.K + k];
        }
        s_sum[g][0][lane] = sum[0];
        __syncthreads();
        if (g != 0 || k >= p.K) return;
        sum[0] = accumulate ? (double)dbias[k] : 0.0;
        for (int j = 0; j < G; ++j) sum[0] += s_sum[j][0][lane];
        dbias[k] = (float)sum[0];
        return;
    }
    const int chunks = 16 * p.P, tile = (int)blockIdx.x / chunks, chunk = (int)blockIdx.x - tile * chunks, jtile = tile / p.kt;
    const int wave = chunk / (4 * p.P), pair = (chunk >> 2) - wave * p.P, v4 = chunk & 3, WC = p.KT == 64 ? 2 : 4;
    const int u0 = 2 * ((wave & (WC - 1)) * p.P + pair), k = (tile - jtile * p.kt) * p.KT + wave / WC * 32 + 8 * v4 + 4 * (lane >> 5);
    if (u0 >= p.units || k - 4 * (lane >> 5) >= p.K) return;
    const float4 *src = reinterpret_cast<const float4 *>(p.part + (size_t)tile * (4096 * p.P) + chunk * 256) + lane;
    const size_t step = (size_t)p.kt * p.jt * (1024 * p.P);
    for (int s = g; s < p.splits; s += G * FLIGHT) {
        float4 v[FLIGHT];
#pragma unroll
        for (int j = 0; j < FLIGHT; ++j) v[j] = s + G * j < p.splits ? src[(size_t)(s + G * j) * step] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int j = 0; j < FLIGHT; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) sum[e] += (double)(&v[j].x)[e];
    }
    if constexpr (G > 1) {
#pragma unroll
        for (int e = 0; e < 4; ++e) s_sum[g][e][lane] = sum[e];
        __syncthreads();
        if (g != 0) return;
        for (int j = 1; j < G; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e) sum[e] += s_sum[j][e][lane];
    }
    const int u = u0 + ((lane >> 4) & 1);
    if (u >= p.units) return;
    const Unit un = unit_of(p, u);
    const Entry en = entry_of(p, jtile * p.subs * 2, un.sub, lane & 15);
    if (en.c >= p.C) return;
    const size_t filter = (size_t)p.C * p.R * p.S;
    float *dst = dw + (size_t)k * filter + (en.c * p.R + en.r) * p.S + un.s;
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (k + e < p.K) {
            float *q = dst + (size_t)e * filter;
            *q = (float)(accumulate ? sum[e] + (double)*q : sum[e]);
        }
}

// Slots that PX pixels and their taps reach at most, so that octets of a pair's two sub-images lie half the banks apart.
int wg_slots(const WgParams &p, int px) {
    const int row_ends = (px - 1 + p.OW - 1) / p.OW, beyond = p.S > p.sx ? p.S - p.sx : 0;
    const int n = (px - 1) * p.sx + row_ends * beyond + p.S;
    return n + (12 - n % 8) % 8;
}

// The tile, the stage and the split of the pixels with the least estimated time.  Nanoseconds of a stage, fitted to launches of 4
// to 59 stages for each workgroup: 55 for each MFMA of a wave (and its neighbour on the SIMD), 264 for a round of staging, 250 for
// the barrier; a partial result is written and read again at 0.6 ns a kilobyte.  On 390 layers (ResNet-18's and drawn) the tile taken
// is 3.6 % behind the fastest in the mean, 21 % at the worst.  Constants that fit better (42, 200, 700 and 0.8: 1.3 % and 16 %) prefer
// stages of 64 pixels where two k-steps are added together, whose error is up to 1.5 times as large (5.7e-8 -> 8.2e-8).
bool wg_plan(WgParams &p, int N, int C, int H, int W, int K, int R, int S, int sh, int sw, int pad, int OH, int OW) {
    const long only = xsmi::option(xsmi::OPT_WGRAD_TILE);      // tests run every tile
    memset(&p, 0, sizeof(p));
    if (R > MAX_TAPS || S > MAX_TAPS) return false;
    p.K = K; p.C = C; p.octets = xsmi::ceil_div(C, 8) * R; p.R = R; p.S = S; p.H = H; p.W = W; p.OH = OH; p.OW = OW; p.OHW = OH * OW;
    p.in_n = C * H * W; p.plane = H * W; p.sh = sh; p.pad = pad; p.M = N * OH * OW; p.N = N; p.dy_next = (K - 1) * p.OHW;
    p.su = S == 1 ? sw : 1; p.sx = S == 1 || OW == 1 ? 1 : sw; p.Wx = (OW - 1) * p.sx + S;
    if (p.Wx >= SMALL_DIV || OH >= SMALL_DIV || H + 2.0 * pad >= 4e6 || W + 2.0 * pad >= 4e6 || (double)p.M >= 1e9) return false;
    // What a tile costs at least: the stages dealt evenly over the chip, one more for every workgroup, one partial result.  The tile
    // of the least is tried first, and most others end at that: a plan takes the host 0.4 to 1.0 us, 1.3 to 1.9 when all are tried.
    struct Tile { int KT, PX, NJ, P, subs, jt, kt, stages; double stage, least; } tile[32];
    int count = 0, first = 0;
    const int all = xsmi::ceil_div(p.octets, 2);
    for (int KT : {64, 32})
        for (int PX : {64, 32}) {
            const int ns = wg_slots(p, PX), y_items = KT / 8 * PX, kt = xsmi::ceil_div(K, KT), stages = xsmi::ceil_div(p.M, PX);
            if (ns > SMALL_PAST) continue;
            const int two = (2 * THREADS - y_items) / (2 * ns), three = (3 * THREADS - y_items) / (2 * ns);
            for (int NJ : {2, 3})
                for (int P : {2, 3, 4, 5}) {
                    if (only && only != KT * 10000 + PX * 100 + P * 10 + NJ) continue;
                    int subs = 256 * P / KT / S;       // units of a tile: 4 P by 64 rows, 8 P by 32
                    if (subs > all) subs = all;
                    if (NJ == 3 && subs <= two) continue;      // two rounds hold as many
                    const int fit = NJ == 3 ? three : two;
                    subs = subs < fit ? subs : fit;
                    if (subs < 1) continue;
                    const int jt = xsmi::ceil_div(all, subs);
                    subs = xsmi::ceil_div(all, jt);    // equal tiles
                    const double rounds = (double)(y_items + 2 * subs * ns) / THREADS;
                    const double stage = 55.0 * P * 6 * (PX / 32) + 264.0 * rounds + 250.0, dealt = (double)kt * jt * stages / 256;
                    tile[count] = {KT, PX, NJ, P, subs, jt, kt, stages, stage, ((dealt > 1.0 ? dealt : 1.0) + 1.0) * stage + (double)kt * jt * P * 16 * 0.6};
                    if (tile[count].least < tile[first].least) first = count;
                    ++count;
                }
        }
    double best = -1.0;
    for (int i = 0; i < count; ++i) {
        const Tile &c = tile[i == 0 ? first : i <= first ? i - 1 : i];
        if (best >= 0 && c.least >= best) continue;
        const int tiles = c.kt * c.jt, once = tiles < 256 ? 256 / tiles : 1;
        int last = 0;
        for (int splits : {once, once / 2, once / 4, once / 8, 512 / tiles, 768 / tiles}) {
            if (splits > 256) splits = 256;
            if (splits > c.stages) splits = c.stages;
            if (splits < 1 || splits == last) continue;
            last = splits;
            if (best >= 0 && tiles * splits <= 256 && (c.stages + splits) * c.stage >= best * splits) continue;
            splits = xsmi::ceil_div(c.stages, xsmi::ceil_div(c.stages, splits));
            const double cost = (double)xsmi::ceil_div(tiles * splits, 256) * (xsmi::ceil_div(c.stages, splits) + 1) * c.stage +
                                (double)tiles * splits * c.P * 16 * 0.6;
            if (best >= 0 && cost >= best) continue;
            best = cost;
            p.KT = c.KT; p.PX = c.PX; p.P = c.P; p.NJ = c.NJ; p.NS = wg_slots(p, c.PX); p.subs = c.subs; p.units = c.subs * S;
            p.kt = c.kt; p.jt = c.jt; p.splits = splits; p.stages = c.stages;
        }
    }
    if (best < 0 || (double)p.splits * p.kt * p.jt * 4096 * p.P * 4 >= 4e9) return false;
    p.per = p.stages / p.splits; p.rem = p.stages % p.splits;
    // Sums of one to a few products: what the bf16 MFMA rounds downwards has no other half of the waves to cancel against, and one
    // fp32 product is rounded to nearest.  `most` products for an element of dw, N for a corner's: error against 64 bits, of that of
    // the fp32 kernels, 1.30 to 1.45 for one product, 1.05 to 1.27 for N = 1 and most = 2 to 4 or N = 2 and most = 2; 0.75 to 1.00
    // for all larger ones (11 filters, 9 maps, N = 1 to 16).  Those few are formed in float64: 480 -> 416, 7 x 7 / 2 at 1 x 1, N=1: 67
    // -> 83 us (fp32 kernels 95); 452 -> 328, 3 x 3 / 2 at 5 x 2, N=1: 16.6 -> 19.7 (19.2).
    const double most = (double)N * (OH < xsmi::ceil_div(H, sh) ? OH : xsmi::ceil_div(H, sh)) * (OW < xsmi::ceil_div(W, sw) ? OW : xsmi::ceil_div(W, sw));
    p.few = N * most <= 4 ? 1 : 0;
    p.x_bytes = (uint32_t)((size_t)N * C * H * W * 4); p.dy_bytes = (uint32_t)((size_t)N * K * OH * OW * 4);
    auto last = [](uint32_t bytes, int plane) { const uint32_t e = (bytes / 4u - 1u) / (uint32_t)plane; return (int)(e < 7u ? e : 7u); };
    p.x_last = last(p.x_bytes, p.plane); p.dy_last = last(p.dy_bytes, p.OHW);
    p.rOW = reciprocal(OW); p.rOHW = reciprocal(p.OHW); p.rWx = reciprocal(p.Wx); p.rOH = reciprocal(OH);
    p.dOW = xsmi::make_fastdiv(OW); p.dOH = xsmi::make_fastdiv(OH);
    p.dNS = xsmi::make_fastdiv(p.NS); p.dR = xsmi::make_fastdiv(R);
    return true;
}

template <int KT, int PX, int P, int NJ>
void wg_launch(const WgParams &p, hipStream_t st) {
    hipLaunchKernelGGL((split_wgrad_kernel<KT, PX, P, NJ>), dim3(p.splits * p.kt * p.jt), dim3(THREADS), 0, st, p);
}
template <int KT, int PX>
void wg_launch(const WgParams &p, hipStream_t st) {
    switch (p.P * 4 + p.NJ) {
    case 2 * 4 + 2: return wg_launch<KT, PX, 2, 2>(p, st);
    case 3 * 4 + 2: return wg_launch<KT, PX, 3, 2>(p, st);
    case 4 * 4 + 2: return wg_launch<KT, PX, 4, 2>(p, st);
    case 5 * 4 + 2: return wg_launch<KT, PX, 5, 2>(p, st);
    case 2 * 4 + 3: return wg_launch<KT, PX, 2, 3>(p, st);
    case 3 * 4 + 3: return wg_launch<KT, PX, 3, 3>(p, st);
    case 4 * 4 + 3: return wg_launch<KT, PX, 4, 3>(p, st);
    default: return wg_launch<KT, PX, 5, 3>(p, st);
    }
}

size_t wg_part_bytes(const WgParams &p) { return xsmi::align_up((size_t)p.splits * p.kt * p.jt * 4096 * p.P * sizeof(float), 256); }

}  // namespace

namespace xsmi {

// Where the split pays: kernel and reduction on about 250 layers of ResNet-18 and drawn, 1 to 512 channels, at N = 1 to 64.
//   fewer than 8 channels (5 under filters of five or more across): no.  An octet's other channels are zeros or another
//     tensor's values (4 -> 32, 3 x 3 at 64 x 64, N=16: 20 -> 25 us; 6 -> 64, 7 x 7 / 2 at 112 x 112, N=32: 80 -> 64).
//   1 x 1: where the fp32 kernels have only the table-driven one, and 4096 results (96 -> 160 at 60 x 60, N=16: 59 -> 40 us; 20 ->
//     40: 20 -> 24; 64 -> 256 at 56 x 56, N=32, on the tap kernel: 44 -> 70).
//   channels and filters multiples of 64, on the tap kernel: from 512 pixels and 2.5e8 products on (64 -> 64 at 56 x 56, N=1: 13
//     -> 17 us; 512 -> 512 at 3 x 3, N=32: 32 -> 34, at 7 x 7: 90 -> 65; 128 -> 256, 3 x 3 / 2 at 28 x 28: N=4 equal, N=32 47 -> 45;
//     64 -> 128, 3 x 3 / 2 at 56 x 56, N=32: 43 -> 47, at half of the error).
//   everything else: yes (32 -> 16, 7 x 7 at 109 x 109, N=5: 179 -> 53 us; 314 -> 32, 3 x 3 / 2 at 95 x 95, N=18: 288 -> 86).  Below
//     3e6 products equal in the mean (81 layers, up to a third slower: 288 -> 15, 7 x 7 / 2 at 4 x 2, N=7: 9.2 -> 12.2) at half of the
//     fp32 kernels' error.
static bool split_wgrad_pays(int C, int K, int R, int S, double pixels) {
    if (C < (S < 5 ? 8 : 5)) return false;
    const bool tap = C % 64 == 0 && K % 64 == 0;
    if (R * S == 1) return !tap && C * K >= 4096;
    return !tap || (pixels >= 512 && pixels * C * K * R * S >= 2.5e8);
}

// Whether the call takes this path, and its plan.
static bool split_wgrad_serves(WgParams &p, int N, int C, int H, int W, int K, int R, int S, int sh, int sw, int pad, bool bf16) {
    const long opt = option(OPT_CONV_SPLIT);
    const int OH = (H + 2 * pad - R) / sh + 1, OW = (W + 2 * pad - S) / sw + 1;
    if (opt == 0 || (opt < 2 && !split_wgrad_pays(C, K, R, S, (double)N * OH * OW))) return false;
    // Under the bf16 flag, at most a tile of the data gradient a compute unit, channels and filters multiples of 64.  A workgroup here
    // fills a unit's LDS and registers: a data gradient on the tap-major kernel, which is started beside the weight gradient
    // (xsmi_conv2d_bwd), waits and lands on the first units that come free, several of its workgroups on one, where the fp32 tap kernel
    // lets it in (both gradients, split -> tap: 192 -> 384, 5 x 5 / 2 at 38 x 38, N=3: 184 -> 139 us; 256 -> 448, 3 x 3 / 2 at 18 x 18, N=9: 96
    // -> 77; 64 -> 128 at 56 x 56, N=8: 60 -> 48; 64 -> 192, 7 x 7 / 2 at 32 x 56, N=8: 121 -> 134).  With four times as many filters as
    // channels this kernel stays ahead (64 -> 512 at 56 x 56, N=4: 90 us, tap 99).  In order, before a split data gradient, the tap
    // kernel is ahead below 1e9 products at 64 channels (64 -> 64 at 56 x 56: N=4 41 -> 36, N=8 49 -> 47; 128 -> 128 at 28 x 28, N=8: 45 -> 50), behind
    // from there on (128 -> 128 at 28 x 28, N=16: 60 and 67; 256 -> 256 at 14 x 14, N=32: 90 and 102; 512 -> 512 at 7 x 7, N=32: 101 and 115).
    // The table-driven fp32 kernel is too slow for either (64 -> 224 at 56 x 56, N=5: 67 us, table-driven 125).  The rule looks at the
    // flag, so that both ways to ask for a weight gradient give the same bits.
    if (opt < 2 && bf16 && K < 4 * C && C % 64 == 0 && K % 64 == 0 && data_gradient_tiles(N, C, H, W) <= cu_count() &&
        ((double)N * OH * OW * C * K * R * S < 1e9 || bf16_data_gradient_by_taps(N, C, H, W, K, R, S, sh, sw, pad, OH, OW)))
        return false;
    return wg_plan(p, N, C, H, W, K, R, S, sh, sw, pad, OH, OW);
}
static size_t wg_ws_bytes(const WgParams &p) { return wg_part_bytes(p) + align_up((size_t)p.splits * p.K * sizeof(float), 256); }

size_t split_wgrad_ws_bytes(int N, int C, int H, int W, int K, int R, int S, int sh, int sw, int pad, bool bf16) {
    WgParams p;
    return split_wgrad_serves(p, N, C, H, W, K, R, S, sh, sw, pad, bf16) ? wg_ws_bytes(p) : 0;
}

int split_conv_bwd_weight(const float *dy, const float *x, float *dw, float *db, int N, int C, int H, int W, int K, int R, int S, int sh,
                          int sw, int pad, bool bf16, int accumulate, void *workspace, size_t workspace_bytes, bool &served) {
    WgParams p;
    served = split_wgrad_serves(p, N, C, H, W, K, R, S, sh, sw, pad, bf16) && workspace_bytes >= wg_ws_bytes(p);
    if (!served) return XSMI_OK;
    p.dy = dy; p.x = x;
    p.part = (float *)workspace;
    if (db) p.dbpart = (float *)((char *)workspace + wg_part_bytes(p));
    hipStream_t st = stream();
    prof_begin();
    if (p.KT == 64 && p.PX == 64) wg_launch<64, 64>(p, st);
    else if (p.KT == 64) wg_launch<64, 32>(p, st);
    else if (p.PX == 64) wg_launch<32, 64>(p, st);
    else wg_launch<32, 32>(p, st);
    prof_end();
    XSMI_LAUNCH_CHECK("split_wgrad_kernel");
    const int dw_blocks = p.kt * p.jt * 16 * p.P, db_blocks = db ? ceil_div(K, 64) : 0;
    auto reduce = [&](auto kernel, int g) {
        hipLaunchKernelGGL(kernel, dim3(dw_blocks + db_blocks), dim3(64 * g), 0, st, p, dw, db, accumulate, dw_blocks);
    };
    if (p.splits >= 32) reduce(split_wgrad_reduce_kernel<16>, 16);
    else if (p.splits >= 8) reduce(split_wgrad_reduce_kernel<4>, 4);
    else reduce(split_wgrad_reduce_kernel<1>, 1);
    XSMI_LAUNCH_CHECK("split_wgrad_reduce_kernel");
    return XSMI_OK;
}

}  // namespace xsmi
