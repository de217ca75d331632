// fp32 convolution forward and backward-data on the bf16 matrix pipes, without giving up float32 precision.
//
// A float32 value is the sum of three bf16 values EXACTLY: 24 significant bits are 8 + 8 + 8, and each remainder a - bf16(a)
// is representable (rounding to nearest even leaves a signed remainder of at most 15, then 7 bits).  So
//     a b = a0 b0 + (a0 b1 + a1 b0) + (a1 b1 + a0 b2 + a2 b0) + [a1 b2 + a2 b1 + a2 b2]
// where the bracket is at most 2^-24 |a b| (|a1| is at most 2^-8 of a's binade, |a2| 2^-17), half a float32 ulp, and is left
// out: six bf16 MFMAs, whose products are exact and whose sums are float32, stand for one float32 product.  The bf16 pipe
// does sixteen times the work of the fp32 pipe per cycle, so the matrix-bound floor falls to 6/16.  The large products (a0
// b0) and the five small ones have accumulators of their own: the chain that carries the rounding of the full sum then has
// one addition per 16 channels and tap, against one per product pair on the fp32 pipe.
//
// What the split does not carry: infinities (inf - inf in a remainder), values within a bf16 rounding of the largest float,
// and the last bits of values below 2^-110.  The first two make the sums that they touch non-finite, the third are looked
// for and given a NaN (split3.h); such sums are formed again in float64 (form_again).
//
// Work layout.  Rows = output channels (64 per tile), columns = output pixels in NCHW order (256 per tile, 128 in small
// launches), 2 x 4 (2 x 2) waves of 32 rows x 64 pixels; passes of at most 32 rows 1 x 8 such waves (sp_plan_tiled).  Waves of
// 64 x 64 halve the conversion and the LDS reads for a product, but their accumulators and fragments spill (128 -> 128 at 28 x
// 28, N=256: 305 -> 342 us; the loop runs 1.22 PFLOP/s of bf16 products there, a large library product 1.30).  The reduction is
// a list of steps (phase, 16 input channels, tap).  A PHASE is a set of taps that read one sub-lattice of the input.  Stride 1:
// all taps; stride 2: the taps of one row and column parity; or, where the input rows of all taps together would not fit the
// LDS, those of as many filter rows as do (216 -> 2, 5 x 5 at 32 x 32, N=52, in images of 3 and 2 rows instead of five of one:
// 202 -> 162 us).  An LDS image holds a phase, in the 128 x 128 tiling several phases and channel groups (SpKind).  In the phase's
// own coordinates the walk has stride 1, so a tile needs one run of positions ("slots") of a grid of pitch Wp = OX + taps
// across - 1, and a tap is nothing but an offset into the run.  The run is staged once per 16 channels for all taps of the
// phase: float32 values are fetched through registers (lanes = slots, eight channels per lane), split there, and written to
// the LDS as [piece][octet][slot][8 channels], so a fragment read is 32 consecutive 16-byte slots whatever the tap is.  The
// LDS image serves up to nine taps, which is what pays for the conversion (ten vector instructions per two values: seven
// split, three look for small ones). The filter is laid out split already, one 6 KB block per step ([piece][octet][row][8]);
// each wave fetches its fragments straight into registers three steps ahead (the waves of a workgroup read the same block at
// about the same time: L1), so the loop has no barrier except around the image of a channel group.
//
// Scheduling is the even split of conv_tap_sk.hip (small launches deal tiles instead, sp_deal_tiles): the steps of all tiles in
// a row are dealt over the resident workgroups; a workgroup whose range starts inside a tile hands its accumulators to the one
// that holds the tile's first step, which adds them in ascending order (bounded wait, deterministic sums).  Row tiles vary
// slowest, so that an XCD's workgroups read few filter blocks.
#include "conv_store.h"
#include "split3.h"

#include <string.h>

namespace {

using xsmi::floatx16;
using xsmi::bf16x8;
using xsmi::uint32x4;
using xsmi::IC;
using xsmi::carried;
typedef uint32_t uint32x2 __attribute__((ext_vector_type(2)));

constexpr int SP_ROWS = 64;                          // rows of a filter block
// Tilings: WR x WC waves of 32 rows x 64 pixels, slots of an LDS image, most workgroups of a launch, whether an image has parts.
struct SpTiling {
    int wr, wc, slots, max_grid;
    bool parts;
    constexpr int rows() const { return 32 * wr; }
    constexpr int pixels() const { return 64 * wc; }
    constexpr int threads() const { return 64 * wr * wc; }
};
constexpr SpTiling SP_TILINGS[] = {{2, 2, 384, 512, false}, {2, 4, 512, 256, false}, {1, 8, 768, 256, false}, {4, 2, 768, 256, true}};
constexpr int sp_block(int pieces) { return pieces * 2 * SP_ROWS * 16; }   // bytes of a step's filter block
constexpr int SP_BLOCK = sp_block(3);
constexpr int SP_MAX_CLASSES = 4, SP_MAX_PHASES = 16;
constexpr bool sp_scratch_holds() {
    for (const SpTiling &k : SP_TILINGS)
        if ((size_t)k.max_grid * 4 > xsmi::SK_SCRATCH_FLAG_BYTES || (size_t)k.max_grid * k.rows() * k.pixels() * 4 > xsmi::SK_SCRATCH_PART_BYTES) return false;
    return true;
}
static_assert(sp_scratch_holds(), "one flag and one partial tile per workgroup");

struct SpPhase {
    int iy0, ix0;          // input place of slot (row v, column u): (v * sy + iy0, u * sx + ix0)
    int Tx, T;             // taps across, taps in all
    int tap0, step0;       // first tap of the class, first step of the tile
    int stride, span;      // steps between channel groups; slots past the last pixel's own that the taps reach
    int r0, rs, s0, ss;    // filter place of tap (a, b): (r0 + rs a, s0 + ss b)
};
// What one image of the LDS serves: the taps of a phase for one group of channels, or (tilings with parts) those of several phases
// and groups, part g nphase + i being phase i of the image's group g.
struct SpKind {
    int phase0, nphase, T, step0;                    // phases; their taps, first step of the tile
    int groups, inv_nphase;                          // channel groups of an image; 256 / nphase + 1
    uint64_t off_lo, off_hi;                         // slot that tap i reads for slot 0, ten bits each, six in off_lo
};
constexpr int SP_MAX_TAPS = 12;                      // of an image with parts: what off_lo and off_hi hold
struct SpClass {
    int M, rows, OY, OX, os_y, os_x;
    long long os_n, os_k, o_base;
    xsmi::FastDiv dOX, dOY, dWp, dHp, dIT, dTM;      // dIT: steps per tile, dTM: pixel tiles
    int Wp, Hp, sy, sx;
    int phase0, nphase, kind0, nkind, taps, blocks;  // blocks: of SP_ROWS rows
    int part_chunks, inv_part_chunks;                // 64-slot chunks of an image's part; 256 / that + 1
    uint32_t iters, first_unit, end_unit, apk_off;
    xsmi::FastDiv dSH;                               // of a launch that deals tiles: workgroups that share one,
    uint32_t end_group;                              // end of the class's workgroups
};
struct SpTapPlace { uint32_t off, iters, step, T; };  // block of (row tile, group): off + rt iters + step + group T
struct SpParams {
    const float *in, *w, *bias;
    const char *apk;
    float *out;
    uint8_t *mask;
    float *part;
    uint32_t *flags, *err;
    uint32_t in_bytes, out_bytes, apk_bytes, spin_limit;
    uint32_t units, upg, urem;                       // steps in all; per workgroup, remainder
    int N, CH, groups, IH, IW, in_n, plane;          // input channels, their groups of 16, floats per image / plane
    int w_row, w_ch, FS;                             // of the layout launches: floats between rows / channels of the filter, filter width
    int ncls, relu, accumulate, tiling;
    int pieces;                                      // 3, or 1: operands rounded to bf16
    SpClass cls[SP_MAX_CLASSES];
    SpPhase ph[SP_MAX_PHASES];
    SpKind kd[SP_MAX_PHASES];
};
// The layout of one 3 x 3 filter, and as many as a launch takes in its arguments (4 KB).
struct SpPackJob {
    const float *w;
    char *apk;
    uint32_t end_block, row_tiles;                   // end of its workgroups in the launch
    int rows, CH, w_row, w_ch;
    int pieces;
    SpTapPlace tap[9];
};
constexpr int SP_PACK_JOBS = 20;
template <int JOBS>
struct SpPackArgs {
    SpPackJob job[JOBS];
    int count;
};
typedef SpPackArgs<SP_PACK_JOBS> SpPackJobs;
static_assert(sizeof(SpPackJobs) <= 4096, "arguments of one launch");
thread_local SpPackJobs *g_pack_jobs = nullptr;      // where layouts are collected instead of launched (split_pack_collect)

constexpr int AGENT = 16;                            // sc1: past the caches that are not coherent across XCDs

// Eight filter values -> three vectors of eight bf16.
__device__ __forceinline__ void split8(const float (&v)[8], uint32x4 &p0, uint32x4 &p1, uint32x4 &p2) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        uint32_t a, b, c;
        xsmi::split_pair3(v[2 * i], v[2 * i + 1], a, b, c);
        p0[i] = a; p1[i] = b; p2[i] = c;
    }
}
// The same where some value of the wavefront does not split: it is left as it is in the second and third piece, behind a first
// one that makes every sum it enters a NaN.
__device__ __forceinline__ void split8_any(const float (&v)[8], uint32x4 &p0, uint32x4 &p1, uint32x4 &p2) {
    constexpr uint32_t NAN16 = xsmi::NAN_PAIR & 0xffffu;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const bool there_l = xsmi::splits(v[2 * i]), there_h = xsmi::splits(v[2 * i + 1]);
        const uint32_t l = __builtin_bit_cast(uint32_t, v[2 * i]), h = __builtin_bit_cast(uint32_t, v[2 * i + 1]);
        uint32_t a, b, c;
        xsmi::split_pair3(there_l ? v[2 * i] : 0.f, there_h ? v[2 * i + 1] : 0.f, a, b, c);
        if (!there_l) { a |= NAN16; b |= l >> 16; c |= l & 0xffffu; }
        if (!there_h) { a |= NAN16 << 16; b |= h & 0xffff0000u; c |= h << 16; }
        p0[i] = a; p1[i] = b; p2[i] = c;
    }
}
// The value again, from the low halves of its three pieces.
__device__ __forceinline__ double unsplit(uint32_t p0, uint32_t p1, uint32_t p2) {
    auto wide = [](uint32_t bits) { return __builtin_bit_cast(float, bits); };   // (the sums are exact)
    return (double)((p0 & 0x7fffu) > 0x7f80u ? wide(p1 << 16 | (p2 & 0xffffu)) : (wide(p0 << 16) + wide(p1 << 16)) + wide(p2 << 16));
}

// The sums of a segment that the split does not carry (split3.h) are formed again in float64: a step's 16 channels are four
// products deep, a lane has channels 4 (l / 16) .. + 3 of a row and of a pixel.  The filter comes out of its layout, whose pieces are
// the value (split8_any), so the filter itself is not read here either; a tap outside the input multiplies a zero, as the
// reference's padding does.  Every workgroup does this for its own steps.  Forward, ordinary values, NaN throughout, one infinity (and
// by the fp32 kernels), us: 32 x 128 x 28 x 28 -> 256, 3 x 3 / 2: 44, 58, 107 (49, 45, 49); 32 x 64 x 56 x 56 -> 64: 58, 102, 116
// (67); without the test for settled sums 44, 200, 115 and 58, 270, 125.
struct SpSteps { int block, s_first, n, f, grp, tap; };   // filter block, steps of the tile, image kind and first group, tap of the image
__device__ __forceinline__ void form_again(floatx16 &r, const SpParams &p, const SpClass &c, const SpSteps &sg, int row0, int m0, int lane,
                                           __amdgpu_buffer_rsrc_t rin, __amdgpu_buffer_rsrc_t rapk) {
    const int l15 = lane & 15, quarter = lane >> 4;
    int oy[2], ox[2], image[2];
    bool there[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int m = m0 + 16 * j + l15, q = (int)xsmi::fdiv((uint32_t)m, c.dOX), n = (int)xsmi::fdiv((uint32_t)q, c.dOY);
        there[j] = m < c.M;
        ox[j] = m - q * c.OX; oy[j] = q - n * c.OY; image[j] = n * p.in_n;
    }
    xsmi::FormAgain again(r, m0 + (lane & 31) < c.M, lane);
    const int a_lane = ((quarter >> 1) * SP_ROWS + row0 + l15) * 16 + (quarter & 1) * 8;
    uint32_t block = c.apk_off + ((uint32_t)sg.block * c.iters + (uint32_t)sg.s_first) * (uint32_t)SP_BLOCK;
    int f = sg.f, grp = sg.grp, tap = sg.tap;
#pragma unroll 1
    for (int s = 0; s < sg.n; ++s, block += SP_BLOCK) {
        if ((s < 4 || (s & 3) == 0) && again.settled()) break;   // (the test is as long as a step)
        const SpKind &kd = p.kd[f];
        const int g = tap / kd.T;
        int i = kd.phase0, ta = tap - g * kd.T;
        while (ta >= p.ph[i].T) ta -= p.ph[i++].T;
        const SpPhase &ph = p.ph[i];
        const int tb = ta % ph.Tx, ch0 = (grp + g) * 16 + 4 * quarter;
        ta /= ph.Tx;
        double a[4][2], b[4][2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            uint32x2 piece[3];
#pragma unroll
            for (int q = 0; q < 3; ++q)
                piece[q] = __builtin_amdgcn_raw_buffer_load_b64(rapk, a_lane + j * 256 + q * 2 * SP_ROWS * 16, (int)block, 0);
            const int iy = (oy[j] + ta) * c.sy + ph.iy0, ix = (ox[j] + tb) * c.sx + ph.ix0;
            const bool in = there[j] && iy >= 0 && iy < p.IH && ix >= 0 && ix < p.IW;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t place = ((uint32_t)image[j] + (uint32_t)(ch0 + i) * (uint32_t)p.plane + (uint32_t)(iy * p.IW + ix)) * 4u;
                const int bits = __builtin_amdgcn_raw_buffer_load_b32(rin, in && ch0 + i < p.CH ? (int)place : (int)0x80000000u, 0, 0);
                b[i][j] = (double)__builtin_bit_cast(float, bits);
                const int sh = 16 * (i & 1);
                a[i][j] = unsplit(piece[0][i >> 1] >> sh, piece[1][i >> 1] >> sh, piece[2][i >> 1] >> sh);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) again.add(a[i], b[i]);
        const int left = p.groups - grp;
        if (++tap == kd.T * (left < kd.groups ? left : kd.groups)) {
            tap = 0;
            grp += kd.groups;
            if (grp >= p.groups) { grp = 0; ++f; }
        }
    }
    again.take(r, lane);
}

// Where a sign mask is kept, the sign of a pre-activation decides which gradients flow, and one within rounding of zero falls on
// one side or the other with the order of the sums: it moves a whole footprint of the gradients (24 -> 40, 5 x 5 at 45 x 61,
// N=7: 2e-4 to 3e-3 of their norm; of 200 passes of that layer 2 had such a sign on the other side than 64 bits, 12 on the fp32
// kernels).  Pre-activations within 2^-21 of the largest sum around them (the lane's 16 rows by 16 pixels; no sum of layers of
// 64 to 12,544 terms was further than 2^-21.6 from 64 bits) are therefore formed again in float64, and taken from there where
// that changes the sign (none of 400 passes).  About one in a million is that small; it costs its wavefront one sum over all
// its lanes (that layer 28.6 -> 29.3 us without one, 35.6 with one; 512 -> 512 at 7 x 7, N=32: 51.0 -> 52.2, 63.7).  A block
// that has more than four of them is left as it is: its largest sum says nothing about the others.
constexpr int SP_DECIDED = 4;
template <int BATCH>
__device__ __forceinline__ void decide_signs(floatx16 &r, const floatx16 &sum, const SpParams &p, const SpClass &c, const float *bias,
                                             int rb, int row0, int m0, int lane, __amdgpu_buffer_rsrc_t rin, __amdgpu_buffer_rsrc_t rapk) {
    float largest = 0.f;
#pragma unroll
    for (int v = 0; v < 16; ++v) largest = __builtin_fmaxf(largest, __builtin_fabsf(sum[v]));
    // ... of the lane's 16 rows, and of its row of 16 lanes (rotated by 1, 2, 4 and 8)
    auto other = [&](auto ctrl) {
        const int bits = __builtin_bit_cast(int, largest);
        largest = __builtin_fmaxf(largest, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(bits, bits, decltype(ctrl)::value, 15, 15, false)));
    };
    other(IC<0x121>{}); other(IC<0x122>{}); other(IC<0x124>{}); other(IC<0x128>{});
    const float bound = largest * 0x1p-21f;
    uint32_t near = 0;
#pragma unroll
    for (int v = 0; v < 16; ++v) near |= __builtin_fabsf(r[v]) <= bound && sum[v] != 0.f ? 1u << v : 0u;
    near = m0 + (lane & 31) < c.M ? near : 0u;
    uint64_t lanes = __builtin_amdgcn_ballot_w64(near != 0);
    if (lanes == 0) return;
    int count = __builtin_popcount(near);
#pragma unroll
    for (int i = 1; i < 64; i *= 2) count += __shfl_xor(count, i);
    if (count > SP_DECIDED) return;
    const int ch16 = lane & 15, a_lane = (ch16 >> 3) * SP_ROWS * 16 + (ch16 & 7) * 2;
    for (; lanes != 0; lanes = __builtin_amdgcn_ballot_w64(near != 0)) {
        const int from = __builtin_ctzll(lanes);
        const int v = __builtin_ctz(__builtin_amdgcn_readlane((int)near, from));
        const int row = row0 + 4 * (from >> 5) + 8 * (v >> 2) + (v & 3), m = m0 + (from & 31);
        const int q = (int)xsmi::fdiv((uint32_t)m, c.dOX), n = (int)xsmi::fdiv((uint32_t)q, c.dOY);
        const int oy = q - n * c.OY, ox = m - q * c.OX, image = n * p.in_n;
        // sixteen lanes for the channels of a step, four steps at a time, BATCH of those in flight
        double total = 0.0;
#pragma unroll 1
        for (int f = c.phase0; f < c.phase0 + c.nphase; ++f) {
            const SpPhase &ph = p.ph[f];
            const uint32_t block = c.apk_off + ((uint32_t)rb * c.iters + (uint32_t)ph.step0) * (uint32_t)SP_BLOCK + (uint32_t)(a_lane + row * 16);
            const uint32_t T = (uint32_t)ph.T, Tx = (uint32_t)ph.Tx, steps = T * (uint32_t)p.groups;
            const uint32_t on = 4 / T, by = 4 - on * T, inv = 65536u / Tx + 1;      // x inv >> 16 = x / Tx, at most 961 taps of 31 across
            uint32_t grp = ((uint32_t)lane >> 4) / T, tap = ((uint32_t)lane >> 4) - grp * T;
#pragma unroll 1
            for (uint32_t base = (uint32_t)lane >> 4; base < steps; base += 4 * BATCH) {
                uint32_t piece[BATCH][3];
                int bits[BATCH];
#pragma unroll
                for (int k = 0; k < BATCH; ++k) {
                    const uint32_t step = base + 4u * k, ta = tap * inv >> 16, tb = tap - ta * Tx;
                    const int ch = (int)grp * 16 + ch16, iy = (oy + (int)ta) * c.sy + ph.iy0, ix = (ox + (int)tb) * c.sx + ph.ix0;
                    const bool in = step < steps && ch < p.CH && iy >= 0 && iy < p.IH && ix >= 0 && ix < p.IW;
                    const uint32_t place = ((uint32_t)image + (uint32_t)ch * (uint32_t)p.plane + (uint32_t)(iy * p.IW + ix)) * 4u;
                    bits[k] = __builtin_amdgcn_raw_buffer_load_b32(rin, in ? (int)place : (int)0x80000000u, 0, 0);
#pragma unroll
                    for (int i = 0; i < 3; ++i)
                        piece[k][i] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(
                            rapk, (int)(step < steps ? block + (grp * (uint32_t)ph.stride + tap) * (uint32_t)SP_BLOCK + (uint32_t)(i * 2 * SP_ROWS * 16) : 0x80000000u), 0, 0);
                    grp += on; tap += by;
                    if (tap >= T) { tap -= T; ++grp; }
                }
#pragma unroll
                for (int k = 0; k < BATCH; ++k)
                    total += unsplit(piece[k][0], piece[k][1], piece[k][2]) * (double)__builtin_bit_cast(float, bits[k]);
            }
        }
#pragma unroll
        for (int i = 1; i < 64; i *= 2) total += __shfl_xor(total, i);
        const float again = (float)(total + (bias ? (double)bias[row] : 0.0));
#pragma unroll
        for (int i = 0; i < 16; ++i) r[i] = i == v && lane == from && (again < 0.f) != (r[i] < 0.f) ? again : r[i];
        if (lane == from) near &= near - 1u;
    }
}

// SIGNS: a sign mask is kept (a kernel of its own: the others would pay for the registers of decide_signs, half a microsecond)
// TILES: every tile has workgroups of its own, which divide its steps and then its output (sp_deal_tiles); otherwise the steps of
// all tiles are dealt evenly.
template <int TILING, bool SIGNS, bool TILES, int PIECES>
__global__ void __launch_bounds__(SP_TILINGS[TILING].threads(), 2) split_conv_kernel(SpParams p) {
    constexpr SpTiling TL = SP_TILINGS[TILING];
    constexpr int WC = TL.wc, ROWS = TL.rows(), SP_PIX = TL.pixels(), THREADS = TL.threads();
    constexpr bool PARTS = TL.parts;
    constexpr int CHUNKS = THREADS / 128, NJ = TL.slots / 64 / CHUNKS;    // 64-slot chunks staged at a time, and how often
    constexpr int SP_PLANE = TL.slots * 16;              // bytes of one (piece, octet) plane
    constexpr int SP_IMAGE = 2 * PIECES * SP_PLANE, SP_BLOCK = sp_block(PIECES);
    constexpr uint32_t PART_BYTES = 32 * THREADS * 4;    // a workgroup's partial tile
    __shared__ __attribute__((aligned(16))) unsigned char s_img[2 * SP_IMAGE];
    __shared__ __attribute__((aligned(16))) float s_bias[2][ROWS];
    __shared__ uint32_t s_fail;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wr = wave / WC, wc = wave % WC, h = lane >> 5, l31 = lane & 31;
    const uint32_t G = gridDim.x, g = xsmi::xcd_contiguous_id(blockIdx.x, G);
    auto range_start = [&](uint32_t j) { return j * p.upg + (j < p.urem ? j : p.urem); };
    uint32_t u = 0, u1 = 0;
    uint32_t share = 0, sharers = 1;                   // this workgroup among those of its tile
    if constexpr (TILES) {
        uint32_t ci = 0;
        while (g >= p.cls[ci].end_group) ++ci;
        const SpClass &c = p.cls[ci];
        const uint32_t first = ci == 0 ? 0u : p.cls[ci - 1].end_group, tile = xsmi::fdiv(g - first, c.dSH);
        sharers = c.dSH.d;
        share = g - first - tile * sharers;
        const uint32_t n = xsmi::fdiv(c.iters, c.dSH), rest = c.iters - n * sharers;
        u = c.first_unit + tile * c.iters + share * n + (share < rest ? share : rest);
        u1 = u + n + (share < rest ? 1u : 0u);
    } else {
        u = range_start(g);
        u1 = range_start(g + 1);
    }
    if (t == 0) s_fail = 0;

    const __amdgpu_buffer_rsrc_t rin = __builtin_amdgcn_make_buffer_rsrc((void *)p.in, 0, (int)p.in_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rapk = __builtin_amdgcn_make_buffer_rsrc((void *)p.apk, 0, (int)p.apk_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rpart =
        __builtin_amdgcn_make_buffer_rsrc((void *)p.part, 0, (int)(TL.max_grid * PART_BYTES), 0x00020000);
    const int row0 = (wr & 1) * 32;                    // in the filter block: a tile of 128 rows has two
    const int a_voff = (h * SP_ROWS + row0 + l31) * 16;
    const int octet = wave & 1, chunk0 = wave >> 1;    // this wave stages slots 64 (chunk0 + CHUNKS j) .. + 63 of one octet
    const uint32_t plane4 = (uint32_t)p.plane * 4u;

    // A segment: steps [s_first, s_first + n) of one tile, beginning with tap `tap` of an image of kind f from channel group `grp` on.
    struct Segment {
        int ci, s_first, n, rt, m0, slot0, nslots, f, grp, tap;
    };
    auto slot_of = [&](const SpClass &c, int m) {
        const int q = (int)xsmi::fdiv((uint32_t)m, c.dOX), n_ = (int)xsmi::fdiv((uint32_t)q, c.dOY);
        return (n_ * c.Hp + (q - n_ * c.OY)) * c.Wp + (m - q * c.OX);
    };
    auto segment_at = [&](uint32_t v) {
        Segment sg;
        sg.ci = 0;
        while (sg.ci + 1 < p.ncls && v >= p.cls[sg.ci].end_unit) ++sg.ci;
        const SpClass &c = p.cls[sg.ci];
        const uint32_t ul = v - c.first_unit, tile = xsmi::fdiv(ul, c.dIT);
        sg.s_first = (int)(ul - tile * c.iters);
        sg.n = (int)c.iters - sg.s_first;
        if (sg.n > (int)(u1 - v)) sg.n = (int)(u1 - v);
        const uint32_t rt = xsmi::fdiv(tile, c.dTM);
        sg.rt = (int)rt;
        sg.m0 = (int)(tile - rt * c.dTM.d) * SP_PIX;
        sg.slot0 = slot_of(c, sg.m0);
        const int m_last = sg.m0 + SP_PIX - 1 < c.M ? sg.m0 + SP_PIX - 1 : c.M - 1;
        sg.nslots = slot_of(c, m_last) - sg.slot0 + 1;
        sg.f = c.kind0;
        while (sg.f + 1 < c.kind0 + c.nkind && sg.s_first >= p.kd[sg.f + 1].step0) ++sg.f;
        const SpKind &kd = p.kd[sg.f];
        const int k = sg.s_first - kd.step0, T = PARTS ? kd.T * kd.groups : kd.T, image = k / T;
        sg.grp = PARTS ? image * kd.groups : image;
        sg.tap = k - image * T;
        return sg;
    };
    auto block_row = [&](const SpClass &c, int rt, int wr) {   // a last tile of 65 rows has one filter block: the other half multiplies it too
        if constexpr (ROWS <= SP_ROWS) return rt;
        const int b = rt * (ROWS / SP_ROWS) + (wr >> 1);
        return b < c.blocks ? b : c.blocks - 1;
    };
    auto block_of = [&](uint32_t v) {                  // byte offset of unit v's filter block (any place past the range)
        if (v >= u1) return 0u;
        int ci = 0;
        while (ci + 1 < p.ncls && v >= p.cls[ci].end_unit) ++ci;
        const SpClass &c = p.cls[ci];
        const uint32_t ul = v - c.first_unit, tile = xsmi::fdiv(ul, c.dIT);
        return c.apk_off + ((uint32_t)block_row(c, (int)xsmi::fdiv(tile, c.dTM), wr) * c.iters + (ul - tile * c.iters)) * (uint32_t)SP_BLOCK;
    };
    uint32_t voff[NJ];
    int group_of[NJ];                                  // of an image with parts: group of each chunk, counted from the image's first
    auto place = [&](const Segment &sg, int f) {       // byte offsets of this lane's slots in channel 0
        const SpClass &c = p.cls[sg.ci];
        const SpKind &kd = p.kd[f];
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            int chunk = chunk0 + CHUNKS * j, i = 0;
            if constexpr (PARTS) {
                const int part = chunk * c.inv_part_chunks >> 8;
                group_of[j] = part * kd.inv_nphase >> 8;
                i = part - group_of[j] * kd.nphase;
                chunk -= part * c.part_chunks;
            }
            const SpPhase &ph = p.ph[kd.phase0 + i];
            const int sl = 64 * chunk + lane;
            const uint32_t P = (uint32_t)(sg.slot0 + sl);
            const int q = (int)xsmi::fdiv(P, c.dWp), n_ = (int)xsmi::fdiv((uint32_t)q, c.dHp);
            const int iy = (q - n_ * c.Hp) * c.sy + ph.iy0, ix = ((int)P - q * c.Wp) * c.sx + ph.ix0;
            const bool ok = sl < sg.nslots + ph.span && n_ < p.N && iy >= 0 && iy < p.IH && ix >= 0 && ix < p.IW;
            voff[j] = ok ? (uint32_t)(n_ * p.in_n + iy * p.IW + ix) * 4u : 0x80000000u;
        }
    };
    float pre[NJ][8];
    // always the same number of loads (slots past the run fetch out of range): the waits below count them
    auto load_image = [&](int grp_) {
        auto whole = [&](int j, int ch0) {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                pre[j][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                rin, (int)voff[j], (int)((uint32_t)(ch0 + e) * plane4), 0));
        };
        auto ragged = [&](int j, int ch0) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const bool there = ch0 + e < p.CH;
                pre[j][e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                rin, (int)(there ? voff[j] : 0x80000000u), (int)(there ? (uint32_t)(ch0 + e) * plane4 : 0u), 0));
            }
        };
        const int ch0 = grp_ * 16 + octet * 8;
        if constexpr (PARTS) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int ch = ch0 + 16 * group_of[j];
                if (ch + 8 <= p.CH) whole(j, ch); else ragged(j, ch);
            }
        } else if (ch0 + 8 <= p.CH) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) whole(j, ch0);
        } else {
#pragma unroll
            for (int j = 0; j < NJ; ++j) ragged(j, ch0);
        }
    };
    // the fetched values into an LDS image: a pair of channels at a time, then the three 16-byte pieces
    uint32x4 piece[PIECES];
    xsmi::SmallTest small;
    auto split_one = [&](auto jt, auto it) {
        constexpr int j = decltype(jt)::value, i = decltype(it)::value;
        if constexpr (PIECES == 1) {
            const xsmi::bf16x2 two = {(__bf16)pre[j][2 * i], (__bf16)pre[j][2 * i + 1]};
            piece[0][i] = __builtin_bit_cast(uint32_t, two);
            return;
        } else {
            uint32_t a, b, c;
            if constexpr (i == 0) small = xsmi::SmallTest{};
            small.add(pre[j][2 * i], pre[j][2 * i + 1]);
            xsmi::split_pair3(pre[j][2 * i], pre[j][2 * i + 1], a, b, c);
            piece[0][i] = a; piece[1][i] = b; piece[2][i] = c;
        }
    };
    auto put = [&](auto j, int to) {
        unsigned char *dst = s_img + to + octet * SP_PLANE + (64 * (chunk0 + CHUNKS * j) + lane) * 16;
        if constexpr (PIECES == 3) piece[0][0] = small.found() ? xsmi::NAN_PAIR : piece[0][0];
#pragma unroll
        for (int q = 0; q < PIECES; ++q) *reinterpret_cast<uint32x4 *>(dst + 2 * q * SP_PLANE) = piece[q];
    };
    auto stage = [&](auto j, int to) {
        split_one(j, IC<0>{}); split_one(j, IC<1>{}); split_one(j, IC<2>{}); split_one(j, IC<3>{});
        put(j, to);
    };
    uint32_t a_off = 0;
    int b_rd[2];                                       // this lane's two pixels in an image
    // Three steps of filter fragments and one of pixel fragments in registers.  A step's filter loads are issued while the
    // step three before it multiplies: vector loads return in order, so they also wait for the image's loads in front of
    // them, which come from memory.
    // (With one piece a step is a single product: its pixel fragments are read while the step before multiplies.)
    constexpr int SETS = PIECES == 1 ? 3 : 1;
    bf16x8 fa[3][PIECES], fb[SETS][2][PIECES];         // [step % 3][piece], [step % SETS][pixel block][piece]
    auto load_a = [&](auto par, auto q) {
        fa[par][q] = __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(
                         rapk, a_voff + (int)q * 2 * SP_ROWS * 16, (int)a_off, 0));
    };
    auto load_step = [&](auto par) {
        if constexpr (PIECES == 3) { load_a(par, IC<2>{}); load_a(par, IC<1>{}); }
        load_a(par, IC<0>{});
    };
    auto read_b = [&](auto set, auto q, int off) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
            fb[set][j][q] = *reinterpret_cast<const bf16x8 *>(s_img + b_rd[j] + off + (int)q * 2 * SP_PLANE);
    };
    int t_left = 0, tb = 0, off = 0, Tx = 1, row_end = 0;
    uint64_t off_lo = 0, off_hi = 0;
    auto next_off = [&]() {                            // past the last tap: back to a place inside the image
        if constexpr (PARTS) {
            off_lo = off_lo >> 10 | (off_hi & 1023) << 50;
            off_hi >>= 10;
            off = (int)(off_lo & 1023) * 16;
            return;
        }
        off += ++tb == Tx ? row_end : 16;
        tb = tb == Tx ? 0 : tb;
        off = --t_left == 0 ? 0 : off;
    };
    floatx16 hi[2], lo[2], images[2];                  // images (TILES): large products of the images before this one
    auto mm = [&](auto par, floatx16 (&acc)[2], int qa, int qb) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
            acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[par][qa], fb[par % SETS][j][qb], acc[j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    // One step.  A piece's registers take the next tap's fragments (past a group's last tap: places that are not used), or
    // the filter block three steps ahead, after the piece's last product.  J >= 0: a part of the next image is split and
    // written to the other half of the LDS, a few instructions behind each pair of MFMAs.
    int image = 0;                                     // byte offset of the image that is multiplied
    int a_left = 0;                                    // steps of the segment whose block ahead has not been requested
    uint32_t a_next[3] = {0, 0, 0};                    // blocks of the three steps after the segment
    auto step = [&](auto par, auto jt) {
        constexpr int J = decltype(jt)::value;
        next_off();
        a_off = a_left > 3 ? a_off + (uint32_t)SP_BLOCK : a_left == 3 ? a_next[0] : a_left == 2 ? a_next[1] : a_next[2];
        --a_left;
        if constexpr (PIECES == 1) {
            read_b(IC<(par + 1) % 3>{}, IC<0>{}, image + off);
            mm(par, hi, 0, 0);
            load_a(par, IC<0>{});
            if constexpr (J >= 0) {
                split_one(jt, IC<0>{}); split_one(jt, IC<1>{}); split_one(jt, IC<2>{}); split_one(jt, IC<3>{});
                put(jt, SP_IMAGE - image);
            }
            return;
        } else {
            mm(par, lo, 2, 0);
            load_a(par, IC<2>{});
            if constexpr (J >= 0) split_one(jt, IC<0>{});
            __builtin_amdgcn_sched_barrier(0);
            mm(par, lo, 1, 0);
            if constexpr (J >= 0) split_one(jt, IC<1>{});
            __builtin_amdgcn_sched_barrier(0);
            mm(par, hi, 0, 0);
            read_b(IC<0>{}, IC<0>{}, image + off);
            if constexpr (J >= 0) split_one(jt, IC<2>{});
            __builtin_amdgcn_sched_barrier(0);
            mm(par, lo, 1, 1);
            load_a(par, IC<1>{});
            if constexpr (J >= 0) split_one(jt, IC<3>{});
            __builtin_amdgcn_sched_barrier(0);
            mm(par, lo, 0, 1);
            read_b(IC<0>{}, IC<1>{}, image + off);
            if constexpr (J >= 0) put(jt, SP_IMAGE - image);
            __builtin_amdgcn_sched_barrier(0);
            mm(par, lo, 0, 2);
            load_a(par, IC<0>{});
            read_b(IC<0>{}, IC<2>{}, image + off);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    // The taps of one image.  Written out up to nine: the waits of each step and the places where the next image is
    // staged are then compile-time facts.
    const auto none = IC<-1>{};
    auto run = [&](int taps) {
        read_b(IC<0>{}, IC<0>{}, image + off);
        if constexpr (PIECES == 3) { read_b(IC<0>{}, IC<1>{}, image + off); read_b(IC<0>{}, IC<2>{}, image + off); }
        int staged = 0;
        const auto third = IC<NJ == 3 ? 2 : -1>{};
        do {
            step(IC<0>{}, none);
            if (taps == 1) break;
            step(IC<1>{}, none);
            if (taps == 2) break;
            step(IC<2>{}, none);
            if (taps == 3) break;
            step(IC<0>{}, IC<0>{});
            staged = 1;
            if (taps == 4) break;
            step(IC<1>{}, none);
            if (taps == 5) break;
            step(IC<2>{}, IC<1>{});
            staged = 2;
            if (taps == 6) break;
            step(IC<0>{}, none);
            if (taps == 7) break;
            step(IC<1>{}, third);
            staged = 3;
            if (taps == 8) break;
            step(IC<2>{}, none);
            for (int i = 9; i < taps; i += 3) {
                step(IC<0>{}, none);
                if (i + 1 < taps) step(IC<1>{}, none);
                if (i + 2 < taps) step(IC<2>{}, none);
            }
        } while (false);
        if (staged < 1) stage(IC<0>{}, SP_IMAGE - image);
        if (staged < 2) stage(IC<1>{}, SP_IMAGE - image);
        if constexpr (NJ == 3)
            if (staged < 3) stage(third, SP_IMAGE - image);
    };

    // The workgroup's steps are one stream: a segment's first image and filter blocks are requested while the segment before
    // it is multiplied, and its output stores drain behind the next one's MFMAs.
    Segment sg = segment_at(u), nx = sg;
    place(sg, sg.f);
    load_image(sg.grp);
    a_off = block_of(u);
    load_step(IC<0>{});
    a_off = sg.n > 1 ? a_off + (uint32_t)SP_BLOCK : block_of(u + 1);
    load_step(IC<1>{});
    a_off = sg.n > 2 ? a_off + (uint32_t)SP_BLOCK : block_of(u + 2);
    load_step(IC<2>{});
    stage(IC<0>{}, 0); stage(IC<1>{}, 0);
    if constexpr (NJ == 3) stage(IC<2>{}, 0);
    int turn = 0;                                      // the set that the next step's filter block is in
    int bias_buf = 0;
    while (true) {
        const SpClass &c = p.cls[sg.ci];
        const bool head = sg.s_first == 0, complete = sg.s_first + sg.n == (int)c.iters;
        const uint32_t tile_end = u + (c.iters - (uint32_t)sg.s_first), u_next = u + (uint32_t)sg.n;
        const int m0 = sg.m0, rt = sg.rt, Wp = c.Wp;
        const bool more = !TILES && u_next < u1;
        if (more) nx = segment_at(u_next);
        a_next[0] = block_of(u_next);
#pragma unroll
        for (int i = 1; i < 3; ++i) a_next[i] = more && nx.n > i ? a_next[0] + (uint32_t)(i * SP_BLOCK) : block_of(u_next + i);
        a_left = sg.n;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int m = m0 + wc * 64 + 32 * j + l31;
            b_rd[j] = h * SP_PLANE + (slot_of(c, m < c.M ? m : c.M - 1) - sg.slot0) * 16;
#pragma unroll
            for (int v = 0; v < 16; ++v) { hi[j][v] = 0.f; lo[j][v] = 0.f; }   // (lo: not used with one piece)
            if constexpr (TILES) images[j] = hi[j];
        }
        bias_buf ^= 1;                                 // the other waves may still be reading the one before
        if (p.bias && (TILES || head) && t < ROWS) s_bias[bias_buf][t] = rt * ROWS + t < c.rows ? p.bias[rt * ROWS + t] : 0.f;
        int left = sg.n, f = sg.f, grp = sg.grp, tap = sg.tap;
        while (left > 0) {
            if (turn) {
#pragma unroll
                for (int q = 0; q < PIECES; ++q) {
                    const bf16x8 x = fa[0][q], y = fa[1][q], z = fa[2][q];
                    fa[0][q] = turn == 1 ? y : z;
                    fa[1][q] = turn == 1 ? z : x;
                    fa[2][q] = turn == 1 ? x : y;
                }
            }
            const SpKind &kd = p.kd[f];
            const int there = PARTS ? p.groups - grp < kd.groups ? p.groups - grp : kd.groups : 1, T = kd.T * there;
            const int taps = left < T - tap ? left : T - tap;
            left -= taps;
            if constexpr (PARTS) {
                off_lo = kd.off_lo;
                off_hi = kd.off_hi;
                off = (int)(off_lo & 1023) * 16;
                for (int i = 0; i < tap; ++i) next_off();
            } else {
                Tx = p.ph[kd.phase0].Tx;
                t_left = T - tap;
                tb = tap % Tx;
                off = (tap / Tx * Wp + tb) * 16;
                row_end = (Wp - Tx + 1) * 16;
            }
            tap = 0;
            // the next image, requested while this one is multiplied
            if (left > 0) {
                grp += there;
                if (grp == p.groups) { grp = 0; ++f; place(sg, f); }
            } else if (more) {
                grp = nx.grp;
                place(nx, nx.f);
            } else {
                grp = p.groups;                        // none: channels past the last read zeros
            }
            load_image(grp);
            xsmi::wait_lgkmcnt0();
            xsmi::block_barrier();                     // this image is complete, and nobody reads the other one any more
            run(taps);
            // The MFMA drops what lies below its accumulator's last bits, so the large products of an image add up from zero
            // and enter the sum in one rounding to nearest: error against 64 bits 0.8 of the even deal's.
            if constexpr (TILES)
                if (left > 0) {
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        images[j] += hi[j];
#pragma unroll
                        for (int v = 0; v < 16; ++v) hi[j][v] = 0.f;
                    }
                }
            turn = taps % 3;
            image = SP_IMAGE - image;
        }
        u = u_next;
        // ---- end of the segment ----
        floatx16 acc[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            acc[j] = PIECES == 3 ? hi[j] + lo[j] : hi[j];
            if constexpr (TILES) acc[j] += images[j];
            if constexpr (PIECES == 3) {
                xsmi::CarriedTest test;
#pragma unroll
                for (int v = 0; v < 16; ++v) test.add(acc[j][v]);
                if (__builtin_amdgcn_ballot_w64(!test.all()) != 0)
                    form_again(acc[j], p, c, SpSteps{block_row(c, rt, wr), sg.s_first, sg.n, sg.f, sg.grp, sg.tap}, row0, m0 + wc * 64 + 32 * j, lane, rin, rapk);
            }
        }
        auto finish = [&](floatx16 &r, int wr, int m) {   // a 32 x 32 block of the output
            const float *bias = p.bias ? s_bias[bias_buf] : nullptr;
            if constexpr (SIGNS) {
                const floatx16 sum = r;
#pragma unroll
                for (int v = 0; v < 16; ++v) r[v] += bias ? bias[wr * 32 + 4 * h + 8 * (v >> 2) + (v & 3)] : 0.f;
                decide_signs<TILING != 0 ? 8 : 4>(r, sum, p, c, bias ? bias + (wr >> 1) * SP_ROWS : nullptr, block_row(c, rt, wr),
                                                  (wr & 1) * 32, m, lane, rin, rapk);
                bias = nullptr;
            }
            xsmi::store_block_32x32(r, c, p.out, p.out_bytes, SIGNS || PIECES == 1 ? p.mask : nullptr, bias, p.relu, p.accumulate, rt * ROWS, ROWS,
                                    wr * 32, m, lane);
        };
        if (TILES ? sharers > 1 : !head) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                uint32x4 q;
#pragma unroll
                for (int e = 0; e < 4; ++e) { const float val = acc[i >> 2][4 * (i & 3) + e]; q[e] = __builtin_bit_cast(uint32_t, val); }
                __builtin_amdgcn_raw_buffer_store_b128(q, rpart, t * 16, (int)(g * PART_BYTES + (uint32_t)i * (THREADS * 16u)), AGENT);
            }
            xsmi::wait_vmcnt<0>();                     // written through, this thread's ...
            __syncthreads();                           // ... and everybody else's
            if (!TILES && t == 0) __hip_atomic_store(p.flags + g, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if constexpr (TILES) {
            if (sharers == 1) {
#pragma unroll
                for (int j = 0; j < 2; ++j) finish(acc[j], wr, m0 + wc * 64 + 32 * j);
                return;
            }
            // Every part is in the scratch memory; the tile's 32 x 32 blocks are dealt over the waves of its workgroups, each of
            // which adds a block's parts in ascending order, all of them at once.  The first workgroup's flag counts who has
            // arrived, then who has read; the last one clears it.
            uint32_t *count = p.flags + (g - share);
            if (t == 0) {
                __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                uint32_t spins = 0;
                bool there = false;
                while (p.spin_limit != 0u &&
                       !(there = __hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= sharers) && ++spins < p.spin_limit)
                    __builtin_amdgcn_s_sleep(1);
                if (!there) {                          // give up, as below
                    s_fail = 1u;
                    __hip_atomic_store(p.err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                }
            }
            __syncthreads();
            if (s_fail) return;
            const uint32_t block = share + sharers * (uint32_t)wave;
            const bool mine = block < 2u * (THREADS / 64);
            const int bw = (int)(block >> 1), bj = (int)(block & 1);
            double sum[16];                            // in float32 a dozen parts would cost up to half as much error again
            if (mine) {
                constexpr uint32_t DEPTH = 4;          // parts in flight
                uint32x4 part[DEPTH][4];
                auto fetch = [&](auto d, uint32_t i) {
#pragma unroll
                    for (int k = 0; k < 4; ++k)
                        part[d][k] = __builtin_amdgcn_raw_buffer_load_b128(
                            rpart, (bw * 64 + lane) * 16, (int)((g - share + i) * PART_BYTES + (uint32_t)(bj * 4 + k) * (THREADS * 16u)), AGENT);
                };
                auto add = [&](auto d) {
#pragma unroll
                    for (int v = 0; v < 16; ++v) {
                        const uint32_t bits = part[d][v >> 2][v & 3];
                        sum[v] += (double)__builtin_bit_cast(float, bits);
                    }
                };
#pragma unroll
                for (int v = 0; v < 16; ++v) sum[v] = -0.0;   // the sum of negative zeros is one
                for (uint32_t i = 0; i < sharers; i += DEPTH) {
                    fetch(IC<0>{}, i);
                    if (i + 1 < sharers) fetch(IC<1>{}, i + 1);
                    if (i + 2 < sharers) fetch(IC<2>{}, i + 2);
                    if (i + 3 < sharers) fetch(IC<3>{}, i + 3);
                    add(IC<0>{});
                    if (i + 1 < sharers) add(IC<1>{});
                    if (i + 2 < sharers) add(IC<2>{});
                    if (i + 3 < sharers) add(IC<3>{});
                }
            }
            __syncthreads();
            if (t == 0 && __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 2 * sharers - 1)
                __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (mine) {
                floatx16 r;
#pragma unroll
                for (int v = 0; v < 16; ++v) r[v] = (float)sum[v];
                finish(r, bw / WC, m0 + bw % WC * 64 + 32 * bj);
            }
            return;
        }
        if (head && !complete) {
            // the rest of the tile was multiplied by the workgroups that follow: a lane waits for each of them, then their
            // parts are added in ascending order, the next one's loads in flight
            for (uint32_t j = g + 1; j < G && range_start(j) < tile_end;) {
                uint32_t np = 1;
                while (np < 64 && j + np < G && range_start(j + np) < tile_end) ++np;
                if ((uint32_t)t < np) {
                    uint32_t spins = 0;
                    bool there = false;
                    while (p.spin_limit != 0u &&
                           !(there = __hip_atomic_load(p.flags + j + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) &&
                           ++spins < p.spin_limit)
                        __builtin_amdgcn_s_sleep(1);
                    if (!there) {                      // give up: the host reports the launch as failed; nothing is stored
                        s_fail = 1u;
                        __hip_atomic_store(p.err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
                    }
                }
                __syncthreads();
                if (s_fail) return;
                uint32x4 part[2][8];
                auto fetch = [&](auto buf, uint32_t i) {
#pragma unroll
                    for (int k = 0; k < 8; ++k)
                        part[buf][k] = __builtin_amdgcn_raw_buffer_load_b128(rpart, t * 16, (int)((j + i) * PART_BYTES + (uint32_t)k * (THREADS * 16u)), AGENT);
                };
                auto add = [&](auto buf) {
#pragma unroll
                    for (int k = 0; k < 8; ++k)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const uint32_t bits = part[buf][k][e];
                            acc[k >> 2][4 * (k & 3) + e] += __builtin_bit_cast(float, bits);
                        }
                };
                fetch(IC<0>{}, 0);
                for (uint32_t i = 0; i < np; i += 2) {
                    if (i + 1 < np) fetch(IC<1>{}, i + 1);
                    add(IC<0>{});
                    if (i + 1 < np) {
                        if (i + 2 < np) fetch(IC<0>{}, i + 2);
                        add(IC<1>{});
                    }
                }
                __syncthreads();                       // everybody has read the parts before their flags are cleared
                if ((uint32_t)t < np) __hip_atomic_store(p.flags + j + (uint32_t)t, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                j += np;
            }
        }
        if (head) {
#pragma unroll
            for (int j = 0; j < 2; ++j) finish(acc[j], wr, m0 + wc * 64 + 32 * j);
        }
        if (!more) break;
        sg = nx;
    }
}

// The filter in its steps' blocks.  A thread owns a row and an octet of channels; lanes are consecutive rows, so a
// wavefront writes whole kilobytes.
// 3 x 3: all nine taps of the octet in registers (each filter line is fetched once; 512 -> 512: 16 -> 6 us against a
// thread per tap, whose 16-byte writes were scattered); every place a tap goes to is in the table `tap`.  A launch of its own
// is 5 to 10 us of fetching its first instructions and lines, whatever the layer's size, so the layouts that are made ahead
// of a step share launches (ResNet-18 step, 33 layouts in two launches: 56 x 56 images 2776 -> 2713 us, 224 x 224 3707 -> 3611).
template <int JOBS>
__global__ void __launch_bounds__(64) split_pack9_kernel(SpPackArgs<JOBS> jobs) {
    int ji = 0;
    while (JOBS > 1 && ji + 1 < jobs.count && blockIdx.x >= jobs.job[ji].end_block) ++ji;
    const SpPackJob &p = jobs.job[ji];
    const uint32_t block = blockIdx.x - (ji ? jobs.job[ji - 1].end_block : 0u);
    const uint32_t o = block / p.row_tiles, rt = block - o * p.row_tiles, row = rt * SP_ROWS + threadIdx.x;
    const int rows = p.rows;
    float v[9][8];
    xsmi::SplitTest test;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        const int ch = (int)o * 8 + e;
        const bool there = (int)row < rows && ch < p.CH;
        const float *src = p.w + (there ? (size_t)row * p.w_row + (size_t)ch * p.w_ch : 0);
#pragma unroll
        for (int t = 0; t < 9; ++t) { v[t][e] = there ? src[t] : 0.f; test.add(v[t][e]); }
    }
    auto put = [&](int t, const uint32x4 &q0, const uint32x4 &q1, const uint32x4 &q2) {
        const SpTapPlace &w = p.tap[t];
        const uint32_t step = rt * w.iters + w.step + (o >> 1) * w.T;
        char *dst = p.apk + w.off + (size_t)step * sp_block(p.pieces) + ((o & 1) * SP_ROWS + threadIdx.x) * 16;
        *reinterpret_cast<uint32x4 *>(dst) = q0;
        if (p.pieces == 1) return;
        *reinterpret_cast<uint32x4 *>(dst + 2 * SP_ROWS * 16) = q1;
        *reinterpret_cast<uint32x4 *>(dst + 4 * SP_ROWS * 16) = q2;
    };
    uint32x4 q0, q1, q2;
    if (p.pieces == 1 || __builtin_amdgcn_ballot_w64(!test.all()) == 0) {
#pragma unroll
        for (int t = 0; t < 9; ++t) { split8(v[t], q0, q1, q2); put(t, q0, q1, q2); }
        return;
    }
    // rolled up and from memory once more: with a choice for each value in the loop above the layout of 64 -> 64 took 9.7 us
    // instead of 6.3, most of it for instructions fetched for the first time
#pragma unroll 1
    for (int t = 0; t < 9; ++t) {
        float u[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int ch = (int)o * 8 + e;
            u[e] = (int)row < rows && ch < p.CH ? p.w[(size_t)row * p.w_row + (size_t)ch * p.w_ch + t] : 0.f;
        }
        split8_any(u, q0, q1, q2);
        put(t, q0, q1, q2);
    }
}
__global__ void __launch_bounds__(256) split_pack_kernel(SpParams p, char *apk) {
    for (int ci = 0; ci < p.ncls; ++ci) {
        const SpClass &c = p.cls[ci];
        const uint32_t rows = (uint32_t)((c.rows + SP_ROWS - 1) / SP_ROWS * SP_ROWS), octets = 2u * (uint32_t)p.groups;
        const uint32_t total = rows * octets * (uint32_t)c.taps;
        for (uint32_t i = blockIdx.x * 256 + threadIdx.x; i < total; i += gridDim.x * 256) {
            const uint32_t row = i % rows, rest = i / rows, o = rest / (uint32_t)c.taps;
            const int tap = (int)(rest - o * (uint32_t)c.taps);
            int f = c.phase0;
            while (f + 1 < c.phase0 + c.nphase && tap >= p.ph[f + 1].tap0) ++f;
            const SpPhase &ph = p.ph[f];
            const int tl = tap - ph.tap0, a = tl / ph.Tx, b = tl - a * ph.Tx;
            const float *src = p.w + (ph.r0 + ph.rs * a) * p.FS + ph.s0 + ph.ss * b;
            float v[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int ch = (int)o * 8 + e;
                v[e] = (int)row < c.rows && ch < p.CH ? src[(size_t)row * p.w_row + (size_t)ch * p.w_ch] : 0.f;
            }
            uint32x4 q0, q1, q2;
            if (p.pieces == 1) split8(v, q0, q1, q2); else split8_any(v, q0, q1, q2);
            const uint32_t step = (row / SP_ROWS) * c.iters + (uint32_t)ph.step0 + (o >> 1) * (uint32_t)ph.stride + (uint32_t)tl;
            char *dst = apk + c.apk_off + (size_t)step * sp_block(p.pieces) + ((o & 1) * SP_ROWS + row % SP_ROWS) * 16;
            *reinterpret_cast<uint32x4 *>(dst) = q0;
            if (p.pieces == 1) continue;
            *reinterpret_cast<uint32x4 *>(dst + 2 * SP_ROWS * 16) = q1;
            *reinterpret_cast<uint32x4 *>(dst + 4 * SP_ROWS * 16) = q2;
        }
    }
}

// slots that the tiles of a class need at most
long sp_slots(int pix, int OY, int OX, int ty, int tx) {
    const long wp = OX + tx - 1, hp = OY + ty - 1;
    const long row_ends = (pix - 1 + OX - 1) / OX, image_ends = ((long)pix - 1 + (long)OX * OY - 1) / ((long)OX * OY);
    return pix + row_ends * (wp - OX) + image_ends * (hp - OY) * wp + (ty - 1) * wp + tx - 1;
}

// Adds a class whose taps are r = r0 + rs a (a < R), s = s0 + ss b (b < S), reading input place (y sy + iy(r), ...), split
// into phases of sub-lattice taps; false if the tables or the LDS image do not hold it.
struct SpTaps { int R, S, r0, rs, s0, ss, iy0, ix0; };            // tap (a, b) reads (y sy + iy0 + a, x sx + ix0 + b)
bool sp_add_class(SpParams &p, int &nph, int &nkd, uint32_t &steps_bytes, const SpTaps &k, int M, int rows, int OY, int OX, int sy, int sx) {
    if (p.ncls == SP_MAX_CLASSES || k.R < 1 || k.S < 1) return false;
    SpClass &c = p.cls[p.ncls];
    const int ny = sy < k.R ? sy : k.R, nx = sx < k.S ? sx : k.S;
    // all rows of a sub-lattice in one image when it fits, otherwise as many at a time as do
    const int ty_max = (k.R + ny - 1) / ny, tx_max = (k.S + nx - 1) / nx;
    const SpTiling &tl = SP_TILINGS[p.tiling];
    if (tl.rows() < SP_ROWS && rows > tl.rows()) return false;
    const int pix = tl.pixels();
    int ty = ty_max;
    while (ty > 1 && (sp_slots(pix, OY, OX, ty, tx_max) > tl.slots || (tl.parts && ty * tx_max > SP_MAX_TAPS))) --ty;
    if (sp_slots(pix, OY, OX, ty, tx_max) > tl.slots || (tl.parts && tx_max > SP_MAX_TAPS)) return false;
    // no more rows than the images need: seven in threes are 3 + 3 + 1, in images of 3 + 2 + 2 no fewer, but shorter ones
    const int images = (ty_max + ty - 1) / ty;
    ty = (ty_max + images - 1) / images;
    int nphase = 0;
    for (int i = 0; i < ny; ++i) nphase += ((k.R - i + ny - 1) / ny + ty - 1) / ty;
    nphase *= nx;
    if (nph + nphase > SP_MAX_PHASES) return false;
    c.phase0 = nph; c.nphase = nphase; c.taps = k.R * k.S;
    c.M = M; c.rows = rows; c.OY = OY; c.OX = OX; c.sy = sy; c.sx = sx;
    c.Wp = OX + tx_max - 1; c.Hp = OY + ty - 1;
    int tap = 0;
    for (int i = 0; i < ny; ++i)
        for (int first = i; first < k.R; first += ny * ty)        // filter rows first, first + ny, ...: at most ty
            for (int j = 0; j < nx; ++j) {
                SpPhase &f = p.ph[nph++];
                const int left = (k.R - first + ny - 1) / ny, na = left < ty ? left : ty, nb = (k.S - j + nx - 1) / nx;
                f.iy0 = k.iy0 + first; f.ix0 = k.ix0 + j;
                f.Tx = nb; f.T = na * nb;
                f.tap0 = tap; f.span = (na - 1) * c.Wp + nb - 1;
                f.r0 = k.r0 + k.rs * first; f.rs = k.rs * ny; f.s0 = k.s0 + k.ss * j; f.ss = k.ss * nx;
                tap += f.T;
            }
    // images: a phase and a group of channels each, or as many of both as make up to nine taps
    const int chunks = xsmi::ceil_div((int)sp_slots(pix, OY, OX, ty, tx_max), 64), parts = tl.parts ? tl.slots / 64 / chunks : 1;
    c.part_chunks = chunks; c.inv_part_chunks = 256 / chunks + 1;
    c.kind0 = nkd;
    int step = 0;
    for (int f = c.phase0; f < nph;) {
        SpKind &kd = p.kd[nkd++];
        kd.phase0 = f; kd.nphase = 0; kd.T = 0; kd.step0 = step;
        do {
            kd.T += p.ph[f].T; ++kd.nphase; ++f;
        } while (f < nph && kd.nphase < parts && kd.T + p.ph[f].T <= 9);
        kd.groups = parts / kd.nphase;
        if (kd.groups > 9 / kd.T) kd.groups = 9 / kd.T;
        if (kd.groups < 1) kd.groups = 1;
        kd.inv_nphase = 256 / kd.nphase + 1;
        int within = 0, n = 0;
        for (int i = kd.phase0; i < f; ++i) { p.ph[i].step0 = step + within; p.ph[i].stride = kd.T; within += p.ph[i].T; }
        for (int part = 0; tl.parts && part < kd.groups * kd.nphase; ++part) {
            const SpPhase &ph = p.ph[kd.phase0 + part % kd.nphase];
            for (int t = 0; t < ph.T; ++t, ++n)
                (n < 6 ? kd.off_lo : kd.off_hi) |= (uint64_t)(part * chunks * 64 + t / ph.Tx * c.Wp + t % ph.Tx) << 10 * (n % 6);
        }
        step += kd.T * p.groups;
    }
    c.nkind = nkd - c.kind0;
    c.iters = (uint32_t)step;
    const int tiles_m = xsmi::ceil_div(M, pix), tiles_r = xsmi::ceil_div(rows, tl.rows()), blocks_r = xsmi::ceil_div(rows, SP_ROWS);
    c.blocks = blocks_r;
    c.dOX = xsmi::make_fastdiv(OX); c.dOY = xsmi::make_fastdiv(OY); c.dWp = xsmi::make_fastdiv(c.Wp); c.dHp = xsmi::make_fastdiv(c.Hp);
    c.dIT = xsmi::make_fastdiv(c.iters); c.dTM = xsmi::make_fastdiv(tiles_m);
    c.apk_off = steps_bytes;
    const double bytes = (double)steps_bytes + (double)blocks_r * c.iters * sp_block(p.pieces), units = (double)p.units + (double)tiles_m * tiles_r * c.iters;
    if (bytes >= 2e9 || units >= 1e9 || (double)c.Wp * c.Hp * p.N >= 1e9) return false;
    steps_bytes += (uint32_t)blocks_r * c.iters * (uint32_t)sp_block(p.pieces);
    c.first_unit = p.units;
    p.units += (uint32_t)tiles_m * (uint32_t)tiles_r * c.iters;
    c.end_unit = p.units;
    ++p.ncls;
    return true;
}

// Steps that a workgroup of a launch has at least.  In a launch that does not fill the chip n steps for each workgroup cost
// 0.45 us n, and the workgroup that adds a tile of I steps together about 0.9 us for each of the I / n - 1 others; the sum is
// smallest at n = sqrt(2 I).
uint32_t sp_least(const SpParams &p) {
    uint32_t steps = 0, least = 4;
    for (int i = 0; i < p.ncls; ++i) steps = p.cls[i].iters > steps ? p.cls[i].iters : steps;
    while (least * least < 2 * steps) ++least;
    return least;
}

// Steps from which a strided pass takes the 128 x 128 tiling: below, its quarter as many workgroups bound the launch.
constexpr uint32_t SP_STRIDED_UNITS = 3300;

bool sp_parts(int CH, int R, int S, int sh, int sw) { return (sh > 1 || sw > 1) && R * S <= 9 && CH >= 64; }

bool sp_fills_rows(int rows, const SpTiling &k) { return 4 * rows >= 3 * xsmi::ceil_div(rows, k.rows()) * k.rows(); }   // three quarters

// The tiling of a pass of m pixels (of its largest class), and its plan.
//   256-pixel tiles stage 2.0 values for each pixel of a 3 x 3 layer's tile where 128-pixel tiles stage 3.0; passes below 1024
//   pixels keep the smaller tile, whose last one is emptier by less.
//   At most 32 rows leave half of a 64-row tile's matrix work to zeros: tiles of 32 x 512 instead, where 64 x 256 would fill the
//   chip (44 x 64 -> 16, 83 x 83: 139 -> 87 us; 10 x 448 -> 5, 5 x 5 at 66 x 66: 278 -> 161).  Below that the number of
//   workgroups bounds the launch, of which there are then half as many (8 x 160 -> 17 at 12 x 59: 25.7 us, 29.5 in wide tiles).
//   Strided passes of at most nine taps and four groups of channels or more, whose row tiles are three quarters full: 128 x 128.
//   The sub-lattices that the taps of a 3 x 3 / 2 filter read are disjoint, so an image of all of them stages no value twice and
//   serves nine taps, where an image a sub-lattice serves one to four; half as many pixels, so that the four parts fit, for twice
//   as many rows.  Backward-data reads one lattice, with one to four taps a
//   class: there the parts are channel groups.  128 -> 256 at 28 x 28, N=32: forward 58 -> 41 us, backward-data 70 -> 47 (fp32
//   kernels 48 and 49); at N=128 147 -> 98 and 215 -> 124 (153, 154).
template <typename Plan>
bool sp_plan_tiled(SpParams &p, int pieces, long m, int rows, bool parts, const Plan &plan) {
    auto as = [&](int tiling) {
        memset(&p, 0, sizeof(p));
        p.tiling = tiling;
        p.pieces = pieces;
        return plan(p);
    };
    if (parts && sp_fills_rows(rows, SP_TILINGS[3]) && as(3) && p.units >= SP_STRIDED_UNITS) return true;
    if (m < 1024) return as(0);
    if (!as(1)) return false;
    if (rows > SP_TILINGS[2].rows() || p.units < 256u * sp_least(p)) return true;
    return as(2) || as(1);
}

bool sp_plan_fwd(SpParams &p, int N, int C, int H, int W, int K, int R, int S, int sh, int sw, int pad, int OH, int OW) {
    return sp_plan_tiled(p, 3, (long)N * OH * OW, K, sp_parts(C, R, S, sh, sw), [&](SpParams &p) {
        p.N = N; p.CH = C; p.groups = xsmi::ceil_div(C, 16); p.IH = H; p.IW = W; p.in_n = C * H * W; p.plane = H * W;
        p.w_row = C * R * S; p.w_ch = R * S; p.FS = S;
        int nph = 0, nkd = 0;
        const SpTaps k = {R, S, 0, 1, 0, 1, -pad, -pad};
        if (!sp_add_class(p, nph, nkd, p.apk_bytes, k, N * OH * OW, K, OH, OW, sh, sw)) return false;
        SpClass &c = p.cls[0];
        c.os_n = (long long)K * OH * OW; c.os_k = (long long)OH * OW; c.o_base = 0; c.os_y = OW; c.os_x = 1;
        p.in_bytes = (uint32_t)((size_t)N * C * H * W * 4); p.out_bytes = (uint32_t)((size_t)N * K * OH * OW * 4);
        return true;
    });
}

// backward-data: a class per residue (h mod sh, w mod sw); taps in ascending order of the dy row they read
bool sp_plan_bwd(SpParams &p, int pieces, int N, int C, int H, int W, int K, int R, int S, int sh, int sw, int pad, int OH, int OW) {
    return sp_plan_tiled(p, pieces, (long)N * H * W / (sh * sw), C, sp_parts(K, R, S, sh, sw), [&](SpParams &p) {
        p.N = N; p.CH = K; p.groups = xsmi::ceil_div(K, 16); p.IH = OH; p.IW = OW; p.in_n = K * OH * OW; p.plane = OH * OW;
        p.w_row = R * S; p.w_ch = C * R * S; p.FS = S;
        int nph = 0, nkd = 0;
        for (int ph = 0; ph < sh && ph < H; ++ph) {
            const int r0 = (ph + pad) % sh, T = r0 < R ? xsmi::ceil_div(R - r0, sh) : 0, cy = (ph + pad - r0) / sh;
            for (int pw = 0; pw < sw && pw < W; ++pw) {
                const int s0 = (pw + pad) % sw, U = s0 < S ? xsmi::ceil_div(S - s0, sw) : 0, cx = (pw + pad - s0) / sw;
                const int OYc = xsmi::ceil_div(H - ph, sh), OXc = xsmi::ceil_div(W - pw, sw);
                const SpTaps k = {T, U, r0 + sh * (T - 1), -sh, s0 + sw * (U - 1), -sw, cy - (T - 1), cx - (U - 1)};
                if (!sp_add_class(p, nph, nkd, p.apk_bytes, k, N * OYc * OXc, C, OYc, OXc, 1, 1)) return false;
                SpClass &c = p.cls[p.ncls - 1];
                c.os_n = (long long)C * H * W; c.os_k = (long long)H * W; c.o_base = (long long)ph * W + pw;
                c.os_y = sh * W; c.os_x = sw;
            }
        }
        p.in_bytes = (uint32_t)((size_t)N * K * OH * OW * 4); p.out_bytes = (uint32_t)((size_t)N * C * H * W * 4);
        return true;
    });
}

// Small launches: every tile has workgroups of its own, n steps each, and all of them add the tile's parts, a block of 32 x 32 a
// wave.  Dealt evenly, the workgroup with a tile's first step adds the others' parts alone, 1.8 us each (64 KB by one compute
// unit): 512 -> 512 at 7 x 7, N=1 22.1 -> 15.1 us, 64 -> 64 at 56 x 56, N=1 16.4 -> 13.6, 448 -> 407, 3 x 3 / 2 at 15 x 15, N=2
// 48 -> 26; 180 layers, both passes, 0.79 of the time.  The stamps of a launch of nine steps a workgroup: parameters 1.6
// us, image 1.5, steps 4.4, parts written 2.1, the others waited for 1.0, parts added 1.5, output 0.4.
// The grid, 0 where the even deal is estimated to be faster.  Times in twentieths of a microsecond beside what both have, fitted to
// those layers (the rule's choice is within 4 % of the best n): a step 8, an image begun 20, parts 20, 4 for each sharer and 80 for
// 256 workgroups; the even deal 200 and 10 a step.  n is tried at the smallest that the resident
// workgroups hold, at whole images and at even parts of one.
uint32_t sp_deal_tiles(SpParams &p, uint32_t res, uint32_t even_grid) {
    uint32_t tiles[SP_MAX_CLASSES], taps[SP_MAX_CLASSES], total = 0, longest = 0, steps = 1;
    bool equal[SP_MAX_CLASSES];                        // images of one length
    for (int i = 0; i < p.ncls; ++i) {
        const SpClass &c = p.cls[i];
        uint32_t images = 0;
        for (int k = c.kind0; k < c.kind0 + c.nkind; ++k) images += (uint32_t)xsmi::ceil_div(p.groups, p.kd[k].groups);
        equal[i] = images * (uint32_t)p.kd[c.kind0].T * (uint32_t)p.kd[c.kind0].groups == c.iters;
        tiles[i] = (c.end_unit - c.first_unit) / c.iters;
        taps[i] = (c.iters + images - 1) / images;
        total += tiles[i];
        if (c.iters > longest) { longest = c.iters; steps = taps[i]; }
    }
    if (res > 256) res = 256;                          // 512 small workgroups write twice the parts (8 x 512 -> 512 at 7 x 7: 26.8 us, 22.5)
    if (total > res) return 0;
    auto grid_of = [&](uint32_t n) {
        uint32_t groups = 0;
        for (int i = 0; i < p.ncls; ++i) groups += tiles[i] * ((p.cls[i].iters + n - 1) / n);
        return groups;
    };
    uint32_t best = 0, best_time = 200 + 10 * ((p.units + even_grid - 1) / even_grid);
    auto attempt = [&](uint32_t n) {
        const uint32_t groups = grid_of(n);
        if (groups > res) return;
        uint32_t time = 0;
        for (int i = 0; i < p.ncls; ++i) {
            const uint32_t iters = p.cls[i].iters, sharers = (iters + n - 1) / n, most = (iters + sharers - 1) / sharers, T = taps[i];
            const bool whole = equal[i] && iters % sharers == 0 && (most % T == 0 || T % most == 0);
            uint32_t images = most / T + (whole ? most < T : most == 1 ? 1 : 2);
            if (images > (iters + T - 1) / T) images = (iters + T - 1) / T;
            const uint32_t cost = 8 * most + 20 * images + (sharers > 1 ? 20 + 4 * sharers + 80 * groups / 256 : 0);
            if (cost > time) time = cost;
        }
        if (time < best_time) { best_time = time; best = n; }
    };
    uint32_t n = (p.units + res - 1) / res;
    if (n < 2) n = 2;
    while (grid_of(n) > res) ++n;
    attempt(n);
    for (uint32_t k = 1; k <= 4; ++k)
        if (steps % k == 0 && steps / k > n) attempt(steps / k);
    for (uint32_t k = (n + steps - 1) / steps, end = k + 3; k < end; ++k) attempt(k * steps);
    attempt(longest);
    if (best == 0) return 0;
    uint32_t groups = 0;
    for (int i = 0; i < p.ncls; ++i) {
        SpClass &c = p.cls[i];
        const uint32_t sharers = (c.iters + best - 1) / best;
        groups += tiles[i] * sharers;
        c.dSH = xsmi::make_fastdiv(sharers);
        c.end_group = groups;
    }
    return groups;
}

int sp_launch_pack(SpPackJobs &jobs) {
    if (jobs.count == 0) return XSMI_OK;
    const dim3 grid(jobs.job[jobs.count - 1].end_block);
    if (jobs.count == 1) {                             // 4 KB of arguments cost a launch by itself 2 us
        hipLaunchKernelGGL(split_pack9_kernel<1>, grid, dim3(64), 0, xsmi::stream(), SpPackArgs<1>{{jobs.job[0]}, 1});
    } else {
        hipLaunchKernelGGL(split_pack9_kernel<SP_PACK_JOBS>, grid, dim3(64), 0, xsmi::stream(), jobs);
    }
    jobs.count = 0;
    XSMI_LAUNCH_CHECK("split_pack9_kernel");
    return XSMI_OK;
}

int sp_run(SpParams &p, int opts, void *workspace) {
    hipStream_t st = xsmi::stream();
    p.apk = (const char *)workspace;
    if (!(opts & 2)) {
        int taps = 0;
        for (int i = 0; i < p.ncls; ++i) taps += p.cls[i].taps;
        const uint32_t row_tiles = (uint32_t)xsmi::ceil_div(p.cls[0].rows, SP_ROWS), octets = 2u * (uint32_t)p.groups;
        if (taps == 9 && p.FS == 3) {
            SpPackJobs own;
            own.count = 0;
            SpPackJobs &jobs = g_pack_jobs ? *g_pack_jobs : own;
            if (jobs.count == SP_PACK_JOBS)
                if (const int rc = sp_launch_pack(jobs)) return rc;
            SpPackJob &job = jobs.job[jobs.count];
            job.w = p.w; job.apk = (char *)workspace; job.row_tiles = row_tiles;
            job.end_block = row_tiles * octets + (jobs.count ? jobs.job[jobs.count - 1].end_block : 0u);
            job.rows = p.cls[0].rows; job.CH = p.CH; job.w_row = p.w_row; job.w_ch = p.w_ch; job.pieces = p.pieces;
            for (int i = 0; i < p.ncls; ++i)
                for (int f = p.cls[i].phase0; f < p.cls[i].phase0 + p.cls[i].nphase; ++f)
                    for (int t = 0; t < p.ph[f].T; ++t) {
                        const SpPhase &ph = p.ph[f];
                        const int r = ph.r0 + ph.rs * (t / ph.Tx), q = ph.s0 + ph.ss * (t % ph.Tx);
                        job.tap[3 * r + q] = SpTapPlace{p.cls[i].apk_off, p.cls[i].iters, (uint32_t)(ph.step0 + t), (uint32_t)ph.stride};
                    }
            ++jobs.count;
            if (!g_pack_jobs)
                if (const int rc = sp_launch_pack(jobs)) return rc;
        } else {
            uint32_t blocks = row_tiles * octets * (uint32_t)p.cls[0].taps / 4 + 1;
            if (blocks > 4096) blocks = 4096;
            hipLaunchKernelGGL(split_pack_kernel, dim3(blocks), dim3(256), 0, st, p, (char *)workspace);
            XSMI_LAUNCH_CHECK("split_pack_kernel");
        }
    }
    if (opts & 4) return XSMI_OK;
    constexpr int TILINGS = sizeof(SP_TILINGS) / sizeof(SP_TILINGS[0]);
    static int resident[6 * TILINGS] = {};
    const SpTiling &tl = SP_TILINGS[p.tiling];
    const int threads = tl.threads();
#define XSMI_SP_KERNELS(SIGNS, TILES, PIECES)                                                                                      \
    split_conv_kernel<0, SIGNS, TILES, PIECES>, split_conv_kernel<1, SIGNS, TILES, PIECES>, split_conv_kernel<2, SIGNS, TILES, PIECES>, \
        split_conv_kernel<3, SIGNS, TILES, PIECES>
    void (*const kernels[6 * TILINGS])(SpParams) = {                  // the tilings of a form; a form's tiles are two forms on
        XSMI_SP_KERNELS(false, false, 3), XSMI_SP_KERNELS(true, false, 3), XSMI_SP_KERNELS(false, true, 3), XSMI_SP_KERNELS(true, true, 3),
        XSMI_SP_KERNELS(false, false, 1), XSMI_SP_KERNELS(false, true, 1)};
#undef XSMI_SP_KERNELS
    auto resident_groups = [&](int which) {
        int &res = resident[which];
        if (res == 0) {
            int per_cu = 0;
            const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernels[which], threads, 0);
            if (e != hipSuccess || per_cu < 1) per_cu = 1;
            const int all = per_cu * xsmi::cu_count(), cap = tl.max_grid;
            res = (all > cap ? cap : all < 8 ? 8 : all) & ~7;
        }
        return (uint32_t)res;
    };
    int which = (p.pieces == 1 ? 4 * TILINGS : p.mask ? TILINGS : 0) + p.tiling;
    const int tiles_form = which + (p.pieces == 1 ? TILINGS : 2 * TILINGS);
    const uint32_t least = sp_least(p);
    uint32_t grid = resident_groups(which);
    if (grid > p.units / least) grid = p.units / least;
    if (grid == 0) grid = 1;
    if (const uint32_t groups = sp_deal_tiles(p, resident_groups(tiles_form), grid)) {
        which = tiles_form;
        grid = groups;
    } else {
        p.upg = p.units / grid; p.urem = p.units % grid;
    }
    const int rc = xsmi::check_device_error("split convolution");
    if (rc) return rc;
    const xsmi::SkScratch scr = xsmi::sk_scratch();
    p.part = scr.part; p.flags = scr.flags; p.err = xsmi::device_error_word();
    const long spin = xsmi::option(xsmi::OPT_SK_SPIN_LIMIT);
    p.spin_limit = spin < 0 ? 0u : spin > 0x7fffffffL ? 0x7fffffffu : (uint32_t)spin;
    xsmi::prof_begin();
    hipLaunchKernelGGL(kernels[which], dim3(grid), dim3(threads), 0, st, p);
    xsmi::prof_end();
    XSMI_LAUNCH_CHECK("split_conv_kernel");
    return XSMI_OK;
}

}  // namespace

namespace xsmi {

// Where the split pays, in kernel plus layout time on random layers of 1 to 512 channels and on ResNet-18's at N = 1 to 32
// (`pixels`: outputs of the pass, of one residue class of a strided backward-data).
//   1 x 1 to 3 taps: no.  An image then serves one tap, and its staging costs more than the fp32 kernels' loads (64 -> 128
//     at 28 x 28, N=32: 12.1 -> 19.2 us).
//   fewer than 16 channels: no.  A step multiplies 16, the rest zeros (4 -> 120, 3 x 3 at 102 x 102, N=53: 109 -> 226 us).
//   strided with whole chunks of 32 channels: in the 128 x 128 tiling (sp_plan_tiled), not with emptier row tiles (160 rows,
//     224 -> 160 at 42 x 42, N=17: 73 -> 92 us) or fewer channels (32 -> 296 at 21 x 70, N=35: 37 -> 45); backward-data, whose
//     images have one to four taps of a few groups, by split_plan_pays.  And where one pixel tile holds all pixels: the fp32
//     kernels then have a few workgroups with a long chain each (256 -> 512 at 14 x 14, N=1: 59 -> 42 us).
//   everything else: yes (64 -> 64 at 56 x 56, N=32: 67 -> 52 us; 369 -> 37, 5 x 5 at 76 x 76, N=2, which had only the
//     table-driven kernel: 801 -> 93 us; equal at the smallest sizes, 64 -> 64 at 56 x 56, N=1: 20.2 -> 21.1 us).
static bool split_pays(int CH, int R, int S, int sh, int sw, long pixels) {
    if (option(OPT_CONV_SPLIT) >= 2) return true;        // wherever it applies, for tests and measurements
    if (R * S < 4 || CH < 16) return false;
    return (sh == 1 && sw == 1) || CH % 32 != 0 || pixels <= 256 || sp_parts(CH, R, S, sh, sw);
}
// ... and whether this plan does.  Strided forward (fp32 kernels -> split, of 320 layers, 0.79 of the time in the mean, at most 1.09):
//   not 4 taps over several row tiles, whose phases have a tap each (320 filters, 2 x 2 / 2, 416 x 54 x 8, N=11: 35 -> 46 us; 250, 64 x
//     107 x 107, N=19: 85 -> 95; one row tile, 118, 384 x 65 x 43, N=21: 95 -> 74);
//   filters of one row or column from 8000 steps of 32 and more a tile on (288 -> 448, 5 x 1 / 2 at 13 x 51, N=12, 4680: 39 -> 46; 64 -> 480 at
//     108 x 48, N=14, 20 a tile: 71 -> 77; 448 -> 288, 1 x 5 / 2 at 41 x 41, N=10, 13440: 125 -> 77);
//   with an odd number of 64-row blocks from 38000 block-steps on (192 -> 192 at 23 x 98, N=8, 7992 steps: 46 -> 54; 512 -> 192 at 20 x 73, N=5,
//     8640: 51 -> 64; 128 -> 192 at 33 x 33, N=45, 12960: 84 -> 61; 288 -> 288 at 23 x 59, N=5, 6318: 44 -> 47; 320 -> 416 at 23 x 23: 46 -> 45).
// Strided backward-data (of 190 layers): a tile's steps must pay for its
// start and its stores, and its second 64 rows must not be zeros, of which the fp32 kernels' 64-row tiles have none.
//   From twice the forward's steps on where every tile has a compute unit (384 -> 512 at 46 x 31, N=3: 50 -> 45 us; 128 -> 256 at 28
//     x 28, N=32: 47 -> 44; below, 256 -> 320 at 35 x 35, N=6, 5520 steps: 40 -> 41), from 15000 on where workgroups go from tile to
//     tile (128 -> 320 at 32 x 31, N=45, 15600: 82 -> 75; 448 -> 128 at 18 x 18, N=59, 10944: 68 -> 85);
//   an even number of 64-row blocks (192 -> 128 at 51 x 51, N=13: 51 -> 77; 192 -> 256 at 32 x 32, N=69: 154 -> 192), or seven and
//     more, from 50000 on (448 -> 512 at 45 x 62, N=8: 226 -> 212; 416 -> 224 at 69 x 69, N=8, 37464: 174 -> 179);
//   from 128 filters on (512 -> 64 at 32 x 51, N=55: 192 -> 208), 256 where the last tile is not whole (352 -> 480 at 40 x 40, N=56:
//     667 -> 501; 352 -> 128 at 28 x 49, N=64: 220 -> 246).
static uint32_t sp_tiles(const SpParams &p) {
    uint32_t tiles = 0;
    for (int i = 0; i < p.ncls; ++i) tiles += (p.cls[i].end_unit - p.cls[i].first_unit) / p.cls[i].iters;
    return tiles;
}
static bool split_plan_pays(const SpParams &p, int R, int S, int sh, int sw, long pixels, bool backward) {
    if (option(OPT_CONV_SPLIT) >= 2 || (sh == 1 && sw == 1) || p.CH % 32 != 0 || pixels <= 256) return true;
    if (!SP_TILINGS[p.tiling].parts) return false;
    const int rows = p.cls[0].rows, blocks = p.cls[0].blocks;
    if (!backward) {
        if (R * S == 4 && rows > SP_TILINGS[3].rows()) return false;
        if ((R == 1 || S == 1) && (p.units < 8000 || p.cls[0].iters < 32)) return false;
        return blocks % 2 == 0 || (double)p.units * blocks >= 38000.0;
    }
    if (p.CH < (rows % SP_TILINGS[3].rows() == 0 ? 128 : 256)) return false;
    if (blocks % 2 != 0) return blocks >= 7 && p.units >= 50000;
    return p.units >= (sp_tiles(p) <= (uint32_t)cu_count() ? 2 * SP_STRIDED_UNITS : 15000u);
}

// Workspace bytes of the split form, 0 where it does not serve the geometry or does not pay.
size_t split_fwd_ws_bytes(int N, int C, int H, int W, int K, int R, int S, int sh, int sw, int pad, int OH, int OW) {
    SpParams p;
    if (option(OPT_CONV_SPLIT) == 0 || !split_pays(C, R, S, sh, sw, (long)N * OH * OW)) return 0;
    if (!sp_plan_fwd(p, N, C, H, W, K, R, S, sh, sw, pad, OH, OW) || !split_plan_pays(p, R, S, sh, sw, (long)N * OH * OW, false)) return 0;
    return align_up(p.apk_bytes, 256);
}
size_t split_bwd_data_ws_bytes(int N, int C, int H, int W, int K, int R, int S, int sh, int sw, int pad, int OH, int OW) {
    SpParams p;
    if (option(OPT_CONV_SPLIT) == 0 || sh > R || sw > S) return 0;
    const long pixels = (long)N * ceil_div(H, sh) * ceil_div(W, sw);
    if (!split_pays(K, R, S, sh, sw, pixels)) return 0;
    if (!sp_plan_bwd(p, 3, N, C, H, W, K, R, S, sh, sw, pad, OH, OW) || !split_plan_pays(p, R, S, sh, sw, pixels, true)) return 0;
    return align_up(p.apk_bytes, 256);
}

// Between the two, layouts of 3 x 3 filters (XSMI_CONV_PACK_ONLY) share launches, on the stream that is current when one is full
// and, for the rest, at the end.
void split_pack_collect() {
    static thread_local SpPackJobs jobs;
    jobs.count = 0;
    g_pack_jobs = &jobs;
}
int split_pack_launch(bool launch) {
    SpPackJobs *jobs = g_pack_jobs;
    g_pack_jobs = nullptr;
    return launch && jobs ? sp_launch_pack(*jobs) : XSMI_OK;
}

// Backward-data with operands rounded to bf16: the same kernel with one piece, so one product for six, which reads dy as it
// is and shares small launches' tiles.  Against the tap-major bf16 kernel, which gathers dy for every tap (tap-major -> this one,
// of 500 layers):
//   from 4 taps on (1 x 1, 128 -> 128 at 56 x 56, N=32: 34 -> 45 us).
//   Stride 1, launches of at most a tile a compute unit, whose idle units are what the tap-major kernel loses: yes, 0.14 to 0.95 of
//     the time (512 -> 512 at 7 x 7: N=32 131 -> 33, N=1 110 -> 17; 128 -> 192, 2 x 2 at 29 x 29, N=35: 32 -> 28), but for at most 32 rows
//     of 32 channels (23 -> 32, 4 x 2 at 48 x 48, N=14: 16 -> 18) or of few products: channels times taps of an image from 384 on, from
//     512 in more than 48 tiles (13 -> 96, 4 x 1 at 99 x 199, N=2, two images of two taps: 19 -> 28; 10 -> 64, 4 x 1 at 12 x 87, N=53, 256,
//     109 tiles: 15 -> 21; 4 -> 64, 2 x 2 at 30 x 30, N=68: 15 -> 19; 7 -> 96, 4 x 1 at 22 x 80, N=45, 384, 155 tiles: 24 -> 27; 6 -> 64, 3 x 2 at
//     30 x 30, N=11, 384, 20 tiles: 18 -> 15; 9 -> 128, 2 x 2 at 42 x 35, N=36: 22.4 -> 21.8).
//   Stride 1, not where rows are so long that an image has two or three taps of fewer than 1024 products (37 -> 128, 2 x 2 at 12 x 156,
//     N=32: 27 -> 36; 40 -> 128, 4 x 1 at 14 x 158, N=15: 25 -> 35; 125 -> 288, 2 x 3 at 12 x 127, N=18: 53 -> 60).
//   Stride 1, larger launches: from 64 reduced channels on (506 -> 32 at 32 x 32, N=125: 125 -> 158) where an image serves nine taps
//     or more in row tiles three quarters full (128 -> 128 at 28 x 28, N=128: 94 -> 71; 64 -> 64 at 56 x 56, N=256: 220 -> 160;
//     512 -> 128, 2 x 2 at 42 x 42, N=84: 231 -> 323; 310 -> 160, 1 x 7 at 68 x 46, N=36: 177 -> 202; 249 -> 288 at 50 x 67 without
//     padding, N=15, whose rows make two images: 150 -> 185; 86 -> 64 at 59 x 59, N=36: 54 -> 58), or for at most 32 rows (16 -> 480,
//     2 x 3 at 35 x 59, N=59: 209 -> 72), 256 products of an image and more (18 -> 64, 4 x 1 at 39 x 157, N=28, two images: 31 -> 49).
//   Strided, in the 128 x 128 tiling as in fp32 (64 -> 128 at 56 x 56, N=32, which has 64 rows: 46 -> 54), with more than two taps a
//     class (193 -> 512, 2 x 2 / 2 at 10 x 62, N=100: 62 -> 100): up to a tile a compute unit (128 -> 256 at 28 x 28, N=32: 40 -> 29;
//     192 -> 384 at 27 x 27, N=12: 55 -> 33), to one and a quarter with filters for three quarters of the channels (256 -> 352 at 63 x
//     63, N=5, 312 tiles: 53 -> 49; 476 -> 224 at 68 x 68, N=2, 304: 42 -> 48; 320 -> 320 at 59 x 67, N=4, 384: 51 -> 57), beyond with
//     twice as many filters as channels and whole row tiles (128 -> 256 at 28 x 28, N=128: 100 -> 89; 113 -> 256 at 36 x 36, N=41:
//     51 -> 62; 224 -> 128 at 54 x 54, N=22: 58 -> 108; 384 -> 128 at 48 x 29, N=126: 230 -> 324).
//   Strided, where one pixel tile holds a class of more than one tap (512 -> 352, 2 x 2 / 2 at 32 x 32, N=1: 24 -> 27), but for 32
//     channels to at most 32 rows, as above, or of fewer than 256 pixels (9 -> 32, 3 x 3 / 2 at 12 x 11, N=3: 11.7 -> 14.4; 2 -> 32, 5 x 5 / 2
//     at 10 x 10: 13.7 -> 17.8; 42 -> 32, 3 x 3 / 2 at 6 x 6, N=3: 12.1 -> 14.9; 70 -> 32, 7 x 7 / 2 at 18 x 18: 25.7 -> 21.0).
// The forward stays with the channels-last kernels: its sums have one order, whatever the batch and the form of the result.
static bool split_bf16_plan_pays(const SpParams &p, int sh, int sw, long pixels) {
    const uint32_t tiles = sp_tiles(p), cus = (uint32_t)cu_count();
    const int rows = p.cls[0].rows;
    const bool few = p.CH < 64 && rows <= SP_TILINGS[2].rows();
    if (sh > 1 || sw > 1) {
        int taps = 0;
        for (int i = 0; i < p.ncls; ++i) taps += p.cls[i].taps;
        if (pixels <= 256L * sh * sw) return taps > sh * sw && !few && (p.CH >= 64 || pixels >= 256);
        if (!SP_TILINGS[p.tiling].parts || taps <= 2 * sh * sw) return false;
        return tiles <= cus || (4 * tiles <= 5 * cus && 4 * p.CH >= 3 * rows) || (p.CH >= 2 * rows && rows % SP_TILINGS[3].rows() == 0);
    }
    if (p.cls[0].nphase > 1 && p.cls[0].taps <= 3 * p.cls[0].nphase && p.CH * p.cls[0].taps < 1024 * p.cls[0].nphase) return false;
    if (tiles <= cus)
        return !few && (rows > SP_TILINGS[2].rows() || p.CH * p.cls[0].taps >= (tiles > 48 ? 512 : 384) * p.cls[0].nphase);
    return p.CH >= 64 && ((rows <= SP_TILINGS[2].rows() && p.CH * p.cls[0].taps >= 256 * p.cls[0].nphase) ||
                          (p.cls[0].taps >= 9 * p.cls[0].nphase && (rows <= SP_ROWS || sp_fills_rows(rows, SP_TILINGS[1]))));
}
size_t split_bf16_bwd_data_ws_bytes(int N, int C, int H, int W, int K, int R, int S, int sh, int sw, int pad, int OH, int OW) {
    SpParams p;
    if (option(OPT_CONV_SPLIT) == 0 || !tap_path_ok(K) || sh > R || sw > S || (R * S < 4 && option(OPT_CONV_SPLIT) < 2)) return 0;
    if (!sp_plan_bwd(p, 1, N, C, H, W, K, R, S, sh, sw, pad, OH, OW)) return 0;
    if (option(OPT_CONV_SPLIT) < 2 && !split_bf16_plan_pays(p, sh, sw, (long)N * H * W)) return 0;
    return align_up(p.apk_bytes, 256);
}

int split_conv_fwd(const float *x, const float *w, const float *bias, float *y, uint8_t *mask, int N, int C, int H, int W,
                   int K, int R, int S, int sh, int sw, int pad, int OH, int OW, int relu, int opts, void *workspace) {
    SpParams p;
    if (!sp_plan_fwd(p, N, C, H, W, K, R, S, sh, sw, pad, OH, OW))
        return set_error("split convolution: geometry not served"), XSMI_ERR_INVALID;
    p.in = x; p.w = w; p.bias = bias; p.out = y; p.mask = relu ? mask : nullptr; p.relu = relu;
    return sp_run(p, opts, workspace);
}

int split_conv_bwd_data(const float *dy, const float *w, float *dx, int N, int C, int H, int W, int K, int R, int S, int sh,
                        int sw, int pad, int OH, int OW, int accumulate, int opts, void *workspace, int pieces) {
    SpParams p;
    if (!sp_plan_bwd(p, pieces, N, C, H, W, K, R, S, sh, sw, pad, OH, OW))
        return set_error("split convolution: geometry not served"), XSMI_ERR_INVALID;
    p.in = dy; p.w = w; p.out = dx; p.accumulate = accumulate;
    return sp_run(p, opts, workspace);
}

}  // namespace xsmi
