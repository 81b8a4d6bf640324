// DeepSeek-V4 style expert conversion for gfx950: packed e2m1 codes with one
// e8m0 scale per 1 x 32 block -> e4m3fn codes with one scale per 128 x 128 tile.
//
//   fp4_rebase : lossless re-basing; outer scale = (largest e8m0 of the tile)/64,
//                element = table(code) * 2^(sb - S + 6), cast without clamp.
//   fp4_amax   : the bf16 value table(code) * 2^(sb-127) is formed in registers
//                (exact), then quantised like a 128 x 128 bf16 tile
//                (scale from amax); the bf16 tensor is written only on request.
//
// One workgroup (256 or 512 threads) owns a 128-row x 256-column "super tile" (two scale
// tiles side by side; the fused kernel has a form with four) so that every row segment it touches is a full 128-byte
// line of packed input and 256 bytes of output.  Lane l of a 32-lane half wave
// owns 4 packed bytes (8 elements); lanes 0-15 belong to the left tile, 16-31
// to the right one (the fused kernel has a form with twice that per lane, 16 lanes
// to a row).  The packed tile lives in 16 (8) VGPRs per lane, so HBM is
// read exactly once.
#include <type_traits>
#include <utility>

#include "lowp_device.h"

using namespace lowp;

namespace {

// Threads per workgroup (NT, a template parameter of everything below): 32 lanes cover a row of the super tile, so
// a pass covers NT / 32 rows and a lane makes 128 / (NT / 32) passes.  Measured on config 5: the re-basing kernel
// is 3-5 % faster with 512 threads than with 256, the fused kernel is indifferent (its per-tile set-up weighs
// more when a lane has fewer passes; with 1024 threads both lose 10-20 %).
constexpr int kRebaseThreads = 512;
constexpr int kAmaxThreads = 256;
// The fused kernel where the buffers' alignment lets a lane own two packed words of a row (one scale byte still covers both), which halves its memory
// instructions and the table work per element (us a launch, back to back, one word -> two: 2048 x 7168 6.13 -> 5.41, 7168 x 2048 5.98 -> 5.25, 512 x
// 1024 level, 32768 x 1152 15.4 -> 13.8, 65536 x 7168 132.7 -> 131.9).  One word a lane is left to other alignments and to the form that writes bf16 too.
// Three forms of it, by the super tiles of 128 x 256 there are for the 256 CUs and by the tiles in a row (lp_fp4_to_fp8_amax).  In brackets super tiles; us,
// two tiles a workgroup with the scale bytes handed round / two with a byte load for each / four with the bytes handed round:
// - up to two on every CU, and three with rows of fewer than 16 tiles, the first: 33024 x 512 [516] 6.16 / 6.32 / 6.65, 24576 x 1024 [768] 6.92 / 7.63 / 7.45; longer rows up to three
//   the second: 8960 x 2048 [560] 6.76 / 6.52 / 6.81, 5888 x 3584 [644] 7.40 / 6.73 / 7.02, 2944 x 7168 [644] 8.25 / 7.05 / 7.22, 70 such sizes drawn 0.96 of the time in fours.
// - beyond, four tiles: 57600 x 512 [900] 9.27 / 8.44 / 7.93, 14464 x 2048 [904] 10.64 / 10.37 / 8.11, 4224 x 7168 [924] 11.63 / 10.84 / 8.41, 65536 x 7168 131.1 / 136.2 / 123.4 =
//   5.8 TB/s.  Not with rows of 1024 columns, whose pieces of a workgroup lie a power of two apart, from seven halves to five on every CU: 25600 x 1024 [800] - / 8.35 / 7.73, 28672 x
//   1024 [896] - / 9.15 / 8.41, 30464 x 1024 [952] - / 9.00 / 9.24, 32768 x 1024 [1024] 10.72 / 9.48 / 11.68, 38400 x 1024 [1200] - / 13.4 / 14.2, 41600 x 1024 [1300] 14.85 / 14.40 / 14.38.
// - where four tiles would leave more than a sixteenth empty at the rows' ends, byte loads up to five on every CU: 38400 x 768 [900] 9.70 / 8.52, 23040 x 1280 [900]
//   10.36 / 8.68, 55552 x 768 [1302] 14.49 / 14.20; and handed round again beyond, 174848 x 768 [4098] 39.3 / 40.6.
constexpr int kWideThreads = 512;

// Maximum over the lane's own 128 x 128 tile, from one barrier.  One word a lane (W = 1, two tiles side by side): the 16 lanes of a DPP row belong to
// one tile and the rows of a wave alternate between the tiles, so a wave reduces to one value per tile (DPP within rows, one cross-lane
// exchange between rows r and r + 2).  Two words a lane: 8 lanes of a row belong to a tile, and each of the workgroup's 16 rows of lanes
// leaves an entry per tile.  They meet in `lds`, and a second DPP reduction finishes.
// The caller must put a barrier before it uses `lds` again.
template <int NT, int W, int TILES>
__device__ __forceinline__ uint32_t tile_max_u32(uint32_t m, uint32_t (*lds)[16], int t)
{
    if constexpr (W == 1) {
        static_assert(TILES == 2);
        m = row16_max_u32(m);
        const uint32_t o = (uint32_t)__shfl_xor((int)m, 32);
        m = o > m ? o : m;
        const int half = (t >> 4) & 1;
        if ((t & 47) == 0) lds[half][t >> 6] = m;          // lanes 0 and 16 of every wave
        __syncthreads();
        const int e = t & 15;
        return row16_max_u32(e < NT / 64 ? lds[half][e] : 0u);
    } else {
        static_assert(W == 2 && NT == 128 * TILES);
        auto fold = [&](auto ctrl) {
            const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, decltype(ctrl)::value, 0xF, 0xF, true);
            m = o > m ? o : m;
        };
        auto eight = [&] {
            fold(std::integral_constant<int, 0xB1>());      // quad_perm: lane ^ 1
            fold(std::integral_constant<int, 0x4E>());      // quad_perm: lane ^ 2
            fold(std::integral_constant<int, 0x141>());     // row_half_mirror: the other quad of the 8 lanes
        };
        eight();
        const int tile = (t >> 3) & (TILES - 1);
        if ((t & 7) == 0) lds[tile][t / (8 * TILES)] = m;
        __syncthreads();
        const u32x2 e = *(const u32x2 *)&lds[tile][(t & 7) * 2];
        m = e.x > e.y ? e.x : e.y;
        eight();
        return m;
    }
}

struct Geometry {
    int64_t row0;        // first row of this lane in pass 0
    int64_t colb;        // byte column of this lane's 4 W packed bytes
    int64_t scol;        // scale column of this lane
    int64_t tile;        // index of this lane's tile in the [rows/128, cols/128] grid
    bool active;         // lane's tile exists (the last super tile of a row may have fewer)
};

template <int W = 1, int TILES = 2>
__device__ __forceinline__ Geometry geometry(int64_t super, int64_t supers_c, int64_t cols, int t)
{
    Geometry g;
    // the launchers keep the number of super tiles below 2^31: a 32-bit division instead of the
    // ~150 scalar instructions of a 64-bit one
    const int64_t sr = (uint32_t)super / (uint32_t)supers_c, sc = super - sr * supers_c;
    constexpr int LANES = 16 * TILES / W;           // of a row
    const int64_t col = sc * (128 * TILES) + (t & (LANES - 1)) * (8 * W);      // logical column of the lane's first element
    g.row0 = sr * 128 + t / LANES;
    g.colb = col >> 1;
    g.scol = col >> 5;
    g.active = col < cols;
    g.tile = sr * (cols >> 7) + (col >> 7);
    return g;
}

// XCD-aware workgroup order: hardware deals consecutive workgroup ids to the 8
// XCDs in turn; remapping gives each XCD a contiguous run of super tiles so
// that neighbours sharing scale cache lines sit behind the same L2.
__device__ __forceinline__ int64_t xcd_remap(int64_t b, int64_t per_xcd) { return (b & 7) * per_xcd + (b >> 3); }

__device__ __forceinline__ uint32_t max_u16x2(uint32_t a, uint32_t b)
{
    return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b)));
}

// value of the e2m1 code in the top nibble
__device__ __forceinline__ float fp4_top(uint32_t x) { const f32x2 t = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(x, 1.0f, 3); return t.y; }

// The e4m3 codes of a lane's 8 elements from its packed word and the 8-entry code table of its scale byte (magnitude code ->
// e4m3 code, low four in `lo`): byte permutes look the nibbles up.  Zero magnitudes carry no sign (fp4_pos_zero).
__device__ __forceinline__ u32x2 lookup8(uint32_t w, uint32_t lo, uint32_t hi)
{
    // even elements sit in the low nibbles of the four bytes, odd elements in the high nibbles
    uint32_t ce = __builtin_amdgcn_perm(hi, lo, w & 0x07070707u);
    uint32_t co = __builtin_amdgcn_perm(hi, lo, (w >> 4) & 0x07070707u);
    ce |= (w & 0x08080808u) << 4;
    co |= w & 0x80808080u;
    return u32x2{__builtin_amdgcn_perm(co, ce, 0x05010400u), __builtin_amdgcn_perm(co, ce, 0x07030602u)};
}

// Code table at the scale byte where half a unit, t1 / 2, is the smallest normal e4m3 number's binade: t1 and t3 (the images
// of 1 and 1.5) are given there, the other entries are theirs times powers of two, 8 per power in the code.  Every scale byte
// `up` steps higher has each entry 8 up higher: rounding to e4m3 is the same in every binade of normal numbers, and no
// element's quotient passes 448.  Entries that no element of a block uses may overflow into the entries above them, which are
// larger and so are not used either; entry 0 is zero and stays zero.
struct CodeTable {
    uint32_t lo, hi;
    __device__ __forceinline__ CodeTable(float t1, float t3)
    {
        const uint32_t c = cvt4(t1, t3, 0.0f, 0.0f), b1 = c & 0xFFu, b3 = (c >> 8) & 0xFFu;
        lo = ((b1 - 8u) << 8) | (b1 << 16) | (b3 << 24);
        hi = (b1 + 8u) | ((b3 + 8u) << 8) | ((b1 + 16u) << 16) | ((b3 + 16u) << 24);
    }
    __device__ __forceinline__ u32x2 codes(uint32_t w, int up) const
    {
        const uint32_t u = (uint32_t)up << 3;
        return lookup8(w, lo + __builtin_amdgcn_perm(0u, u, 0x0000000Cu), hi + __builtin_amdgcn_perm(0u, u, 0x00000000u));
    }
};

template <int NT>
__global__ __launch_bounds__(NT) void fp4_rebase(const uint8_t *__restrict__ packed, const uint8_t *__restrict__ scale,
                                                  int64_t cols, int64_t supers_c, int64_t n_supers, int64_t per_xcd,
                                                  uint8_t *__restrict__ q, void *__restrict__ scale_out, int scale_dtype)
{
    constexpr int kRowsPerPass = NT / 32, kPasses = 128 / kRowsPerPass;
    __shared__ uint32_t lds[2][16];
    const int64_t super = xcd_remap(blockIdx.x, per_xcd);
    if (super >= n_supers) return;
    const int t = threadIdx.x;
    const Geometry g = geometry<>(super, supers_c, cols, t);
    const int64_t pcols = cols >> 1, scols = cols >> 5;

    uint32_t w[kPasses];
    uint32_t sb[kPasses];
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
        const int64_t r = g.row0 + p * kRowsPerPass;
        if (g.active) {
            w[p] = __builtin_nontemporal_load((const uint32_t *)(packed + r * pcols + g.colb));
            sb[p] = scale[r * scols + g.scol];
        } else {
            w[p] = 0; sb[p] = 0;
        }
    }
    uint32_t S = 0;
#pragma unroll
    for (int p = 0; p < kPasses; ++p) S = sb[p] > S ? sb[p] : S;
    S = tile_max_u32<NT, 1, 2>(S, lds, t);

    const bool nan_tile = S == 0xFFu;
    if (g.active && (t & 15) == 0 && (t >> 5) == 0) {
        // outer = 2^(S-127) / 64 rounded to e8m0: byte max(S-6, 0); 0xFF stays NaN
        uint32_t ob = nan_tile ? 0xFFu : (S > 6u ? S - 6u : 0u);
        if (scale_dtype == LP_E8M0) ((uint8_t *)scale_out)[g.tile] = (uint8_t)ob;
        else ((float *)scale_out)[g.tile] = e8m0_to_f32(ob);
    }
    if (!g.active) return;

#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
        const int64_t r = g.row0 + p * kRowsPerPass;
        u32x2 out;
        if (!nan_tile) {
            // offset = 2^(sb - S + 6); below 2^-30 every product rounds to (signed) zero anyway
            int d = (int)sb[p] - (int)S + 6;
            d = d < -30 ? -30 : d;
            const float off = u2f((uint32_t)(127 + d) << 23);
            float v[8];
            fp4_decode8(fp4_pos_zero(w[p]), v);
#pragma unroll
            for (int j = 0; j < 8; ++j) v[j] *= off;
            out.x = cvt4(v[0], v[1], v[2], v[3]);
            out.y = cvt4(v[4], v[5], v[6], v[7]);
        } else {
            out.x = 0x7F7F7F7Fu; out.y = 0x7F7F7F7Fu;
        }
        __builtin_nontemporal_store(out, (u32x2 *)(q + r * cols + (g.colb << 1)));
    }
}

// ---------------------------------------------------------------- fused amax

// A whole layer in one launch is bound by HBM; one expert's tensor (a few MB, a launch of its own in a loader's loop) by the
// arithmetic of the two or three waves a SIMD gets, since nothing else covers it: what was 63 vector operations per 8 elements
// is 38 with one conversion for the maximum and the moved code table (W = 1).  us a launch, back to back: 2048 x 7168 6.96 -> 5.85, 512 x
// 1024 4.3 -> 3.8, 65536 x 7168 137.6 -> 135.3 (256 threads; 512 level with it, 1024 behind: 6.6 and 149).

template <class F, int... I>
__device__ __forceinline__ void each(F &&f, std::integer_sequence<int, I...>)
{
    (f(std::integral_constant<int, I>()), ...);
}

template <int W>
__device__ __forceinline__ void store_codes(const u32x2 *out, uint8_t *dst)
{
    if constexpr (W == 2) __builtin_nontemporal_store(u32x4{out[0].x, out[0].y, out[1].x, out[1].y}, (u32x4 *)dst);
    else __builtin_nontemporal_store(out[0], (u32x2 *)dst);
}

template <int MODE, bool WRITE_BF16, int NT, int W, int TILES = 2, bool BYTES = W == 1, bool WAVES = BYTES && W == 2>
__global__ __launch_bounds__(NT) void fp4_amax(const uint8_t *__restrict__ packed, const uint8_t *__restrict__ scale,
                                                int64_t cols, int64_t supers_c, int64_t n_supers, int64_t per_xcd,
                                                float amax_floor, int zero_rule, uint8_t *__restrict__ q,
                                                void *__restrict__ scale_out, int scale_dtype, uint16_t *__restrict__ bf16_out)
{
    constexpr int LANES = 16 * TILES / W, kRowsPerPass = NT / LANES, kPasses = 128 / kRowsPerPass;
    static_assert(W == 1 || !WRITE_BF16);
    __shared__ __attribute__((aligned(8))) uint32_t lds[TILES][16];
    asm volatile("" ::"s"(packed), "s"(scale));              // fetched with the other arguments, not behind the test below
    const int64_t super = xcd_remap(blockIdx.x, per_xcd);
    if (super >= n_supers) return;
    const int t = threadIdx.x;
    const Geometry g = geometry<W, TILES>(super, supers_c, cols, t);
    const int64_t pcols = cols >> 1, scols = cols >> 5;

    // Lanes of a tile past the last one read the super tile's first tile instead, so the loads need no branches; their results
    // are never stored.
    const int place = g.active ? 0 : (t & (LANES - 1)) / (16 / W);
    const int64_t ld_colb = g.colb - place * 64, ld_scol = g.scol - place * 4;
    uint32_t w[kPasses][W];
    uint32_t sb[kPasses];
    uint32_t four = 0;
    // (a load at any address: the scales need not start on a word)
    if constexpr (!BYTES) __builtin_memcpy(&four, scale + (g.row0 + (t & 7) * kRowsPerPass) * scols + (ld_scol & ~3), 4);
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
        const int64_t r = g.row0 + p * kRowsPerPass;
        if constexpr (W == 2) {
            const u32x2 v = __builtin_nontemporal_load((const u32x2 *)(packed + r * pcols + ld_colb));
            w[p][0] = v.x;
            w[p][W - 1] = v.y;
        } else {
            w[p][0] = fp4_pos_zero(__builtin_nontemporal_load((const uint32_t *)(packed + r * pcols + ld_colb)));
        }
        if constexpr (BYTES) sb[p] = scale[r * scols + ld_scol];
        if constexpr (BYTES && W == 2) {
            w[p][0] = fp4_pos_zero(w[p][0]);
            w[p][W - 1] = fp4_pos_zero(w[p][W - 1]);
        }
    }
    if constexpr (!BYTES) {
        // Each of the 8 lanes that share a row of a tile has loaded the row's four scale bytes of one pass; they hand them round.
        static_assert(kPasses == 8);
        const uint32_t shift = (t & 6) * 4;
        auto pass = [&](auto pc) {
            constexpr int p = decltype(pc)::value;
            w[p][0] = fp4_pos_zero(w[p][0]);
            w[p][W - 1] = fp4_pos_zero(w[p][W - 1]);
            int d = __builtin_amdgcn_update_dpp(0, (int)four, 0x150 + p, 0xF, 0x3, false);      // row_newbcast to lanes 0 .. 7 of the row
            d = __builtin_amdgcn_update_dpp(d, (int)four, 0x158 + p, 0xF, 0xC, false);          // ... 8 .. 15
            sb[p] = ((uint32_t)d >> shift) & 0xFFu;
        };
        each(pass, std::make_integer_sequence<int, kPasses>());
    }

    // amax of |table(code)| * 2^(sb-127).  The product is exact in fp32 (and
    // in bf16) for scale bytes 2..252; any other byte sends the whole super
    // tile down the literal slow path.
    // The largest of a word's eight magnitude codes is the largest magnitude: folded in the top nibble of each half and then of
    // the word (what lies below that nibble does not matter to the maximum), so one element of eight is converted.
    float amax_lane = 0.0f;
    uint32_t sb_min = 255u, sb_max = 0u;
#pragma unroll
    for (int p = 0; p < kPasses; ++p) {
        uint32_t h = 0;
#pragma unroll
        for (int j = 0; j < W; ++j) {
            const uint32_t x = w[p][j] & 0x77777777u;
            h = max_u16x2(h, max_u16x2(max_u16x2(x, x << 4), max_u16x2(x << 8, x << 12)));
        }
        const uint32_t h16 = h << 16;
        h = h > h16 ? h : h16;
        amax_lane = fmaxf(amax_lane, fp4_top(h) * u2f(sb[p] << 23));
        sb_min = sb[p] < sb_min ? sb[p] : sb_min;
        sb_max = sb[p] > sb_max ? sb[p] : sb_max;
    }
    const uint32_t mbits = f2u(amax_lane);
    const bool edge = sb_min < 2u || sb_max > 252u;
    // Every thread of the workgroup must take the same number of barriers, so both slow decisions (edge scale bytes, tile scale outside the
    // fast range) are made for the super tile as a whole: an edge byte travels as the key 0xFFFFFFFF (products are finite
    // positive floats, so that pattern is free), and a wave, which holds lanes of every tile, asks whether any of its lanes has a slow one.
    const uint32_t key = tile_max_u32<NT, W, TILES>(edge ? 0xFFFFFFFFu : mbits, lds, t);
    bool slow_tile = __any(key == 0xFFFFFFFFu);
    BlockScale bs;
    // Each element is +-{0, .5, 1, 2, 4} * 2^e (even codes and 0.5) or +-{1, 2, 4} * 1.5 * 2^e (codes
    // 1.5, 3, 6), so its quotient by the tile scale is a power-of-two multiple of one of two numbers,
    // c1 = RN(1/s) and c3 = RN(1.5/s) (resp. f and RN(1.5 f) in the multiply form): two correctly
    // rounded constants per tile replace one division per element, and power-of-two scaling keeps
    // them correctly rounded.
    float c1 = 1.0f, c3 = 1.5f;
    if (!slow_tile) {
        auto out_of_range = [&](const BlockScale &b) -> bool {
            if (MODE == LP_SCALE_POW2) return b.exp2 < -100 || b.exp2 > 100;
            if (MODE == LP_SCALE_DIV) return !b.fast;
            return !(b.div >= 0x1p-100f && b.div <= 0x1p100f);
        };
        bs = derive_scale<MODE>(u2f(key), amax_floor, zero_rule);
        slow_tile = __any(out_of_range(bs));
        if (MODE == LP_SCALE_POW2) {
            c1 = ldexpf(1.0f, -bs.exp2);
            c3 = ldexpf(1.5f, -bs.exp2);
        } else if (MODE == LP_SCALE_DIV) {
            c1 = bs.recip;
            c3 = 1.5f / bs.div;
        } else {
            c1 = bs.div;
            c3 = 1.5f * bs.div;
        }
    }

    // Behind a branch that it knows to be uniform the compiler keeps 30 registers more, which takes two to three of eight waves of a SIMD.  WAVES: the waves
    // instead, for launches of few rounds -- two words with a byte load each, and one word up to five super tiles on every CU (0.95 of the time up to two); larger
    // ones are better off with the registers (one word from 1280 super tiles on 1.03 <- 1; 65536 x 4096 in fours 74.9 <- 80.3).
    uint32_t slow = slow_tile;
    if constexpr (WAVES) asm volatile("" : "+v"(slow));
    if (!slow) {
        if (g.active && (t & (16 / W - 1)) == 0 && t < LANES) store_scale(scale_out, scale_dtype, g.tile, bs.stored);
        if (!g.active) return;
        // All 8 elements of a pass share one scale byte sb, so their codes are eight numbers per pass:
        //   magnitude 0 .5 1 1.5 2 3 4 6  ->  e4m3(0, t1/2, t1, t3, 2 t1, 2 t3, 4 t1, 4 t3),  t = c * 2^(sb-127).
        // Where t1 / 2 is a normal e4m3 number (scale bytes within 11 or so of the largest that counts), the table of the tile
        // moved up by 8 per power of two is that table: two permutes and two additions.
        const uint32_t c1b = f2u(c1), c3b = f2u(c3);
        const int cf = (int)(c1b >> 23);
        const int sb0 = 249 - cf;                                  // c1 * 2^(sb0 - 127) / 2 = 1.x * 2^-6
        if (!WRITE_BF16 && !__any((int)sb_min < sb0)) {
            const uint32_t to5 = (uint32_t)(122 - cf) << 23;       // c1, c3 at sb0
            const CodeTable tab(u2f(c1b + to5), u2f(c3b + to5));
#pragma unroll
            for (int p = 0; p < kPasses; ++p) {
                const int64_t r = g.row0 + p * kRowsPerPass;
                u32x2 out[W];
#pragma unroll
                for (int j = 0; j < W; ++j) {
                    uint32_t wp = w[p][j];
                    asm volatile("" : "+v"(wp));               // keep the packed word, not values derived before the barrier
                    out[j] = tab.codes(wp, (int)sb[p] - sb0);
                }
                store_codes<W>(out, q + r * cols + (g.colb << 1));
            }
            return;
        }
        // Otherwise four conversions build the table of each pass in two registers (a conversion costs about 3 plain VALU
        // instructions, measured).
        // The factors are formed by adding to the exponent field.  c1 and c3 are normal here (exponent
        // field cf, c3's at most cf + 1), so t1/2 .. 4 t3 are normal floats for sb in [129 - cf, 378 - cf],
        // and clamping sb to that range changes no result: a non-zero block has 2^(sb-127) <= 2 amax,
        // i.e. sb <= 264 - cf, so above the range every element is zero (and zero maps to table entry 0);
        // below it every quotient is under 2^-120 in magnitude and becomes a signed zero with the clamped
        // factor as with the true one.
        const int sb_lo = 129 - cf, sb_hi = 378 - cf;
        const uint32_t c1adj = c1b - (127u << 23), c3adj = c3b - (127u << 23);
#pragma unroll
        for (int p = 0; p < kPasses; ++p) {
            const int64_t r = g.row0 + p * kRowsPerPass;
            int sbe = (int)sb[p];
            sbe = sbe < sb_lo ? sb_lo : (sbe > sb_hi ? sb_hi : sbe);
            const uint32_t t1 = c1adj + ((uint32_t)sbe << 23), t3 = c3adj + ((uint32_t)sbe << 23);
            const uint32_t tab_lo = cvt4(0.0f, u2f(t1 - (1u << 23)), u2f(t1), u2f(t3));
            const uint32_t tab_hi = cvt4(u2f(t1 + (1u << 23)), u2f(t3 + (1u << 23)), u2f(t1 + (2u << 23)), u2f(t3 + (2u << 23)));
            u32x2 out[W];
            uint32_t wp = 0;
#pragma unroll
            for (int j = 0; j < W; ++j) {
                wp = w[p][j];
                asm volatile("" : "+v"(wp));                   // keep the packed word, not values derived before the barrier
                out[j] = lookup8(wp, tab_lo, tab_hi);
            }
            store_codes<W>(out, q + r * cols + (g.colb << 1));
            if (WRITE_BF16) {
                const float s = u2f(sb[p] << 23);            // sb in 2..252: a normal power of two
                float b[8];
                fp4_decode8(wp, b);
                u32x4 o = {pack_bf16(b[0] * s, b[1] * s), pack_bf16(b[2] * s, b[3] * s), pack_bf16(b[4] * s, b[5] * s),
                           pack_bf16(b[6] * s, b[7] * s)};
                __builtin_nontemporal_store(o, (u32x4 *)(bf16_out + r * cols + (g.colb << 1)));
            }
        }
        return;
    }

    __syncthreads();                                          // the reduction below writes `lds` again
    // Slow tile: scale bytes at the edge of the e8m0 range (bf16 rounding,
    // overflow to inf, NaN).  Literal arithmetic with software casts; inputs
    // are read again from memory so that the fast path keeps its registers.
    uint32_t m2 = 0;
    if (g.active) {
        for (int i = 0; i < kPasses * W; ++i) {
            const int64_t r = g.row0 + i / W * kRowsPerPass;
            const uint32_t wp = fp4_pos_zero(*(const uint32_t *)(packed + r * pcols + g.colb + i % W * 4));
            const float s = e8m0_to_f32(scale[r * scols + g.scol]);
            for (int j = 0; j < 8; ++j) {
                float b = bf16_bits_to_f32(sw_f32_to_bf16(sw_e2m1_to_f32((wp >> (4 * j)) & 0xFu, false) * s));
                uint32_t a = f2u(b) & 0x7FFFFFFFu;
                m2 = a > m2 ? a : m2;
            }
        }
    }
    m2 = tile_max_u32<NT, W, TILES>(m2, lds, t);
    const bool has_nan = m2 > 0x7F800000u;
    const float amax = u2f(has_nan ? 0x7FC00000u : m2);
    bs = derive_scale<MODE>(amax, amax_floor, zero_rule);
    if (has_nan && MODE == LP_SCALE_DIV) { bs.div = amax; bs.stored = amax; }
    if (g.active && (t & (16 / W - 1)) == 0 && t < LANES) store_scale(scale_out, scale_dtype, g.tile, bs.stored);
    if (!g.active) return;
    for (int i = 0; i < kPasses * W; ++i) {
        const int64_t r = g.row0 + i / W * kRowsPerPass, colb = g.colb + i % W * 4;
        const uint32_t wp = fp4_pos_zero(*(const uint32_t *)(packed + r * pcols + colb));
        const float s = e8m0_to_f32(scale[r * scols + g.scol]);
        uint32_t o0 = 0, o1 = 0, h0 = 0, h1 = 0, h2 = 0, h3 = 0;
        for (int j = 0; j < 8; ++j) {
            uint32_t hb = sw_f32_to_bf16(sw_e2m1_to_f32((wp >> (4 * j)) & 0xFu, false) * s);
            uint32_t c = quant_slow<MODE>(bf16_bits_to_f32(hb), bs);
            uint32_t hs = hb << (16 * (j & 1)), cs = c << (8 * (j & 3));
            if (j < 4) o0 |= cs; else o1 |= cs;
            if (j < 2) h0 |= hs; else if (j < 4) h1 |= hs; else if (j < 6) h2 |= hs; else h3 |= hs;
        }
        if (bf16_out) {
            u32x4 ob = {h0, h1, h2, h3};
            *(u32x4 *)(bf16_out + r * cols + (colb << 1)) = ob;
        }
        u32x2 out = {o0, o1};
        *(u32x2 *)(q + r * cols + (colb << 1)) = out;
    }
}

int check_fp4_args(const char *name, const void *packed, const void *scale, int64_t rows, int64_t cols, const void *q_out,
                   const void *scale_out)
{
    LP_REQUIRE(rows >= 0 && cols >= 0, "%s: bad shape", name);
    LP_REQUIRE(rows % 128 == 0 && cols % 128 == 0, "%s: shape (%lld, %lld) must be a multiple of 128 x 128", name,
               (long long)rows, (long long)cols);
    if (rows == 0 || cols == 0) return 1;
    LP_REQUIRE(packed && scale && q_out && scale_out, "%s: null pointer", name);
    LP_REQUIRE((uintptr_t)packed % 4 == 0 && (uintptr_t)q_out % 8 == 0, "%s: buffers must be 8-byte aligned", name);
    return LP_OK;
}

}  // namespace

extern "C" int lp_fp4_to_fp8_rebase(const void *packed, const void *scale, int64_t rows, int64_t cols, void *q_out,
                                    void *scale_out, int scale_dtype, lp_stream_t stream)
{
    LP_REQUIRE(scale_dtype == LP_E8M0 || scale_dtype == LP_F32, "lp_fp4_to_fp8_rebase: scale_dtype must be LP_E8M0 or LP_F32");
    int rc = check_fp4_args("lp_fp4_to_fp8_rebase", packed, scale, rows, cols, q_out, scale_out);
    if (rc) return rc > 0 ? LP_OK : rc;
    const int64_t supers_c = (cols + 255) / 256, n_supers = (rows / 128) * supers_c;
    const int64_t per_xcd = (n_supers + 7) / 8;
    LP_REQUIRE(per_xcd * 8 <= 0x7FFFFFFF, "lp_fp4_to_fp8_rebase: too many tiles");
    hipLaunchKernelGGL(fp4_rebase<kRebaseThreads>, dim3((unsigned)(per_xcd * 8)), dim3(kRebaseThreads), 0, (hipStream_t)stream, (const uint8_t *)packed,
                       (const uint8_t *)scale, cols, supers_c, n_supers, per_xcd, (uint8_t *)q_out, scale_out, scale_dtype);
    return check_launch("lp_fp4_to_fp8_rebase");
}

extern "C" int lp_fp4_to_fp8_amax(const void *packed, const void *scale, int64_t rows, int64_t cols, int scale_mode,
                                  float amax_floor, int zero_rule, void *q_out, void *scale_out, int scale_dtype,
                                  void *bf16_out, lp_stream_t stream)
{
    LP_REQUIRE(is_scale_dtype(scale_dtype), "lp_fp4_to_fp8_amax: bad scale_dtype %d", scale_dtype);
    LP_REQUIRE(scale_mode >= LP_SCALE_POW2 && scale_mode <= LP_SCALE_MUL, "lp_fp4_to_fp8_amax: bad scale_mode");
    LP_REQUIRE(zero_rule >= LP_ZERO_NONE && zero_rule <= LP_ZERO_SCALE_TO_ONE, "lp_fp4_to_fp8_amax: bad zero_rule");
    LP_REQUIRE(amax_floor >= 0.0f, "lp_fp4_to_fp8_amax: amax_floor must be >= 0");
    int rc = check_fp4_args("lp_fp4_to_fp8_amax", packed, scale, rows, cols, q_out, scale_out);
    if (rc) return rc > 0 ? LP_OK : rc;
    LP_REQUIRE(!bf16_out || (uintptr_t)bf16_out % 16 == 0, "lp_fp4_to_fp8_amax: bf16_out must be 16-byte aligned");
    hipStream_t st = (hipStream_t)stream;
    auto go = [&](auto kernel, int threads, int tiles) -> int {
        const int64_t supers_c = (cols / 128 + tiles - 1) / tiles, n_supers = (rows / 128) * supers_c, per_xcd = (n_supers + 7) / 8;
        LP_REQUIRE(per_xcd * 8 <= 0x7FFFFFFF, "lp_fp4_to_fp8_amax: too many tiles");
        hipLaunchKernelGGL(kernel, dim3((unsigned)(per_xcd * 8)), dim3(threads), 0, st, (const uint8_t *)packed, (const uint8_t *)scale, cols, supers_c,
                           n_supers, per_xcd, amax_floor, zero_rule, (uint8_t *)q_out, scale_out, scale_dtype, (uint16_t *)bf16_out);
        return check_launch("lp_fp4_to_fp8_amax");
    };
    const bool two_words = (uintptr_t)packed % 8 == 0 && (uintptr_t)q_out % 16 == 0;
    // see kWideThreads
    const int64_t per_row = cols / 128, two = (per_row + 1) / 2 * 2, four = (per_row + 3) / 4 * 4, supers = rows / 128 * (two / 2);
    const bool apart = per_row == 8 && 2 * supers > 7 * kCUs && supers <= 5 * kCUs;
    const bool wide = four * 16 <= two * 17 && supers > 3 * kCUs && !apart;
    const bool many = supers > 5 * kCUs, handed = many || supers <= kCUs * (per_row < 16 ? 3 : 2);
#define LAUNCH(MODE)                                                                                                   \
    return bf16_out ? go(fp4_amax<MODE, true, kAmaxThreads, 1>, kAmaxThreads, 2)                                        \
         : !two_words && many ? go(fp4_amax<MODE, false, kAmaxThreads, 1>, kAmaxThreads, 2)                             \
         : !two_words ? go(fp4_amax<MODE, false, kAmaxThreads, 1, 2, true, true>, kAmaxThreads, 2)                      \
         : wide ? go(fp4_amax<MODE, false, kWideThreads, 2, 4>, kWideThreads, 4)                                        \
         : handed ? go(fp4_amax<MODE, false, kAmaxThreads, 2>, kAmaxThreads, 2)                                         \
                  : go(fp4_amax<MODE, false, kAmaxThreads, 2, 2, true>, kAmaxThreads, 2)
    if (scale_mode == LP_SCALE_POW2) LAUNCH(LP_SCALE_POW2);
    if (scale_mode == LP_SCALE_DIV) LAUNCH(LP_SCALE_DIV);
    LAUNCH(LP_SCALE_MUL);
#undef LAUNCH
}
