// Pieces shared by the FP8 GEMM translation units.
#pragma once
#include "lowp_device.h"

namespace lowp {
namespace gemm {

template <int SDT>
__device__ __forceinline__ float scale_at(const void *s, int64_t idx)
{
    if (SDT == LP_F32) return ((const float *)s)[idx];
    // e8m0: 2^(b-127); byte 0 is the fp32 subnormal 2^-127 and 0xFF is NaN
    const uint32_t b = ((const uint8_t *)s)[idx];
    return u2f(b == 0u ? 0x00400000u : (b == 0xFFu ? 0x7FC00000u : b << 23));
}

// Tile order: tiles are numbered so that 32 consecutive numbers form a block of
// 8 M-tiles x 4 N-tiles (shared operand panels), and each XCD (workgroup id
// modulo 8) is handed whole blocks, so panels are re-used out of one L2.
constexpr int GROUP_M = 8, GROUP_N = 4, CHUNK = GROUP_M * GROUP_N;

// Tile `lin` of the numbering.
template <class I>
__device__ __forceinline__ void tile_of(I lin, I tiles_m, I tiles_n, int64_t &tm, int64_t &tn)
{
    // groups of GROUP_M m-tiles (the last may be short); inside a group, blocks of
    // GROUP_N n-tiles (the last may be narrow); inside a block m runs fastest
    const I per_group = GROUP_M * tiles_n;
    const I grp = lin / per_group, in_grp = lin - grp * per_group;
    const I left = tiles_m - grp * GROUP_M;
    const I gm = left < GROUP_M ? left : GROUP_M;
    const I per_nblock = gm * GROUP_N;
    const I nblk = in_grp / per_nblock, in_blk = in_grp - nblk * per_nblock;
    tm = grp * GROUP_M + in_blk % gm;
    tn = nblk * GROUP_N + in_blk / gm;
}

// ends_first: the chunks an XCD works through come alternately from the front and the back of the tile
// list (grid = number of workgroups launched, a multiple of 8 * CHUNK).  Grouped problems list experts in
// caller order; when the heavy experts sit at one end, this keeps compute-bound tiles and tiles that only
// stream weights on the machine at the same time.
// In 32 bits, which hold every grid and so every number here: the divisions stand in front of a workgroup's first request, and in 64 bits they are some
// 150 instructions each (us, 64 / 32 bits: e8m0 844 x 1664 x 1408 9.36 / 9.21, 1857 x 3584 x 1536 15.8 / 15.5; fp32 1000 x 4992 x 2944 26.15 / 25.8).
__device__ __forceinline__ bool tile_coords(uint32_t b, int64_t tiles_m, int64_t tiles_n, int64_t &tm, int64_t &tn,
                                            bool ends_first = false, uint32_t grid = 0)
{
    const uint32_t s = b >> 3, turn = s / CHUNK, Q = grid / (8 * CHUNK);
    const uint32_t q = !ends_first ? turn : (turn & 1) ? Q - 1 - (turn >> 1) : (turn >> 1);
    const uint32_t lin = (q * 8 + (b & 7)) * CHUNK + s % CHUNK;
    if (lin >= (uint32_t)tiles_m * (uint32_t)tiles_n) return false;
    tile_of<uint32_t>(lin, (uint32_t)tiles_m, (uint32_t)tiles_n, tm, tn);
    return true;
}

// Partial sums of a range of K (gemm_asm_split, splitk_reduce): SplitPlan's rows of 128 columns per tile column, a tile's rows behind those of the tile
// above it.  In a tile, a wave's 64 rows x 64 columns in the order it stores them: blocks of 16 columns, in those blocks of 16 rows, 4 columns
// of a row per lane.  With the 16-row blocks of both waves side by side a wave's stores jump by 8 KB: 1024 x 512 x 7168 14.6 -> 18.0 us.  Where there is no
// room for rows beyond M its last ones go by blocks of rows first, so that only the last block's lines are not whole.  In floats,
// which 32 bits number (at most 32 MiB); `rows`: from the tile's first row on.
__device__ __forceinline__ uint32_t partial_tile(uint32_t tm, uint32_t tn, uint32_t rows) { return (tn * rows + tm * 128) * 128; }

__device__ __forceinline__ int partial_offset(int wm, int wn, int nb, int mb, int lane, int rows)
{
    const int left = (rows < 128 ? rows : 128) - wm * 64, own = left < 64 ? left : 64, high = own - mb * 16 < 16 ? own - mb * 16 : 16;
    const int block = own == 64 ? nb * (16 * 64) + mb * (16 * 16) : mb * (16 * 64) + nb * (16 * high);
    return wm * (64 * 128) + wn * (64 * own) + block + ((lane >> 4) * (4 * high) + (lane & 15) * 4);
}

// The tiles of G problems of one shape, numbered problem by problem: pieces of 2^shift consecutive ones are dealt to the XCDs in
// turn, forwards and backwards: in a list sorted by length the XCD with the longest of one turn has the shortest of the next.  (With every problem dealt from XCD 0 on as above, a problem of few tiles ran on few XCDs: 20 weight gradients of 1024 x
// 1408 with three K blocks, 24 tiles each, on one of eight: 131 us, dealt in turn 30.  With pieces that end with their problem, the
// last and smaller ones could all fall to the same XCDs: 32 problems of 1408 x 2048 with
// sixteen K blocks, 48 tiles each, 200 us, across problems 166.)  Workgroup b ->
// problem g and its tile; false: none.  In 32 bits, which hold the grid and so every number here: the divisions stand in front of
// a workgroup's first request, and in 64 bits they took 0.4 us (one problem of 128 x 256 with eight K blocks 6.6 us, so 6.1).
__device__ __forceinline__ bool list_coords(uint32_t b, uint32_t G, uint32_t tiles_m, uint32_t tiles_n, int shift, int64_t &g, int64_t &tm, int64_t &tn)
{
    const uint32_t tiles = tiles_m * tiles_n, s = b >> 3;
    const uint32_t turn = s >> shift, xcd = (b & 7) ^ (turn & 1 ? 7 : 0);
    const uint32_t id = ((turn * 8 + xcd) << shift) + (s & ((1u << shift) - 1)), problem = id / tiles;
    if (problem >= G) return false;
    g = problem;
    tile_of<uint32_t>(id - problem * tiles, tiles_m, tiles_n, tm, tn);
    return true;
}

// Whole chunks, whose operand panels are shared in an L2, where that leaves the XCDs alike, or where every XCD has one and they take
// no more rounds of an XCD's `slots` workgroups (0: not known) than tiles dealt one by one would (2 problems of 2432 x 1280 with eight K
// blocks, 12 chunks: quarters 12.3 us, whole 10.6); a quarter of one otherwise.
inline int list_shift(int64_t G, int64_t tiles_m, int64_t tiles_n, int slots = 0)
{
    static_assert(CHUNK == 1 << 5 && GROUP_M == 1 << 3);
    const int64_t tiles = G * tiles_m * tiles_n, chunks = (tiles + CHUNK - 1) / CHUNK, most = (chunks + 7) / 8;
    if (most * 8 * 4 <= chunks * 5) return 5;
    return slots && chunks >= 8 && (most * CHUNK + slots - 1) / slots <= (tiles + 8 * slots - 1) / (8 * slots) ? 5 : 3;
}

inline int64_t list_grid(int64_t G, int64_t tiles_m, int64_t tiles_n, int shift)
{
    const int64_t round = 8ll << shift;
    return (G * tiles_m * tiles_n + round - 1) / round * round;
}

// Rows of expert e from the caller's offset table, made safe to use: both ends are clamped to [0, M_total] and a
// decreasing pair is an empty expert, so a bad table cannot send a tile outside the operands.
__device__ __forceinline__ int expert_rows(const int32_t *__restrict__ m_offsets, int e, int64_t M_total, int64_t &begin)
{
    int64_t a = m_offsets[e], b = m_offsets[e + 1];
    a = a < 0 ? 0 : (a > M_total ? M_total : a);
    b = b < 0 ? 0 : (b > M_total ? M_total : b);
    begin = a;
    return b > a ? (int)(b - a) : 0;
}

inline int64_t padded_grid(int64_t tiles_m, int64_t tiles_n)
{
    const int64_t chunks = (tiles_m * tiles_n + CHUNK - 1) / CHUNK;
    return ((chunks + 7) / 8) * 8 * CHUNK;
}

// gemm_fp8_big.hip
int choose_big_tn(int64_t M, int64_t N);
int launch_big(const void *Aq, const void *As, const void *Bq, const void *Bs, int scale_dtype, int64_t M, int64_t N,
               int64_t K, void *C, int64_t ldc, int out_dtype, int tn, hipStream_t st);

bool rowscale_asm_ok(const void *As, const void *Bs, int scale_dtype, int64_t M, int64_t N, int64_t K);
int launch_rowscale_asm(const void *Aq, const void *As, const void *Bq, const void *Bs, const int32_t *groups, int G, int max_k_blocks,
                        int multiple, int64_t M, int64_t N, void *C, int out_dtype, hipStream_t st);

// gemm_skinny.hip: at most 64 activation rows
constexpr int kSkinnyBlocks = 7;          // K blocks one workgroup handles
// at most 16 activation rows: one workgroup per 16 weight rows over all of K (gemm_thin.hip)
bool thin_ok(int64_t M, int64_t N, int64_t K);
bool thin_rows_ok(int64_t M, int64_t N, int64_t K);
int launch_thin_rows(const void *Aq, const void *As, const void *Bq, const void *Bs, int scale_dtype, int64_t M, int64_t N, int64_t K,
                     void *C, int out_dtype, hipStream_t st);
// per-row e8m0 scales, problems of one or two K blocks, no K loop (gemm_rowscale_small.hip); groups == nullptr: one problem
int launch_rowscale_small(const void *Aq, const void *As, const void *Bq, const void *Bs, const int32_t *groups, int G, int k_blocks,
                          int64_t M, int64_t N, void *C, int out_dtype, hipStream_t st);
int launch_thin(const void *Aq, const void *As, const void *Bq, const void *Bs, int scale_dtype, int64_t M, int64_t N, int64_t K,
                void *C, int out_dtype, hipStream_t st);
void skinny_plan(int64_t N, int64_t K, int &splits, int &per);
int64_t skinny_workspace_bytes(int64_t N, int splits);
int launch_skinny(const void *Aq, const void *As, const void *Bq, const void *Bs, int scale_dtype, int64_t M, int64_t N,
                  int64_t K, void *C, int out_dtype, float *ws, int splits, int per, hipStream_t st);

int launch_nt_unit_scales(const void *A, const void *B, const void *ones, int64_t M, int64_t N, int64_t K, void *C, int out_dtype,
                          hipStream_t st, bool bf16 = false);
bool nt_unit_scales_ok(const void *ones, int64_t M, int64_t N, int64_t K);
bool wide_keeps(int64_t M, int64_t N, int64_t K);
bool launch_wide(const void *Aq, const void *As, const void *Bq, const void *Bs, int scale_dtype, int64_t M, int64_t N, int64_t K,
                 void *C, int64_t ldc, int out_dtype, hipStream_t st, int *rc);
bool launch_mixed(const void *Aq, const void *As, const void *Bq, const void *Bs, int scale_dtype, int64_t M, int64_t N, int64_t K,
                  int64_t n_big, void *C, int64_t ldc, int out_dtype, hipStream_t st, int *rc);
// A dense problem on 128 x 128 tiles of which those at or behind column n_whole are cut into `splits` ranges of `per` K blocks; rows: of
// partial sums, M or whole tiles; fold: e8m0 products are added up in fp32 (gemm_asm_split).
struct SplitPlan {
    int64_t n_whole;
    int splits, per;
    int64_t rows;
    bool fold;
};
int launch_split(const void *Aq, const void *As, const void *Bq, const void *Bs, int scale_dtype, int64_t M, int64_t N, int64_t K,
                 const SplitPlan &plan, void *C, int out_dtype, float *ws, hipStream_t st);
bool mid_asm_ok(const void *As, const void *Bs, int scale_dtype, int64_t M, int64_t N, int64_t K);
int launch_mid_asm(const void *Aq, const void *As, const void *Bq, const void *Bs, int scale_dtype, int64_t M, int64_t N,
                   int64_t K, void *C, int64_t ldc, int out_dtype, hipStream_t st);
bool big_grouped_ok(const void *As, const void *Bs, int scale_dtype, int64_t M_total, int64_t N, int64_t K);
bool grouped_nn_ok(const void *As, const void *Bs, int scale_dtype, int E, int64_t M_total, int64_t N, int64_t K);
int launch_grouped_nn(const void *Aq, const void *As, const void *Bq, const void *Bs, const int32_t *m_offsets, int E,
                      int64_t M_total, int64_t N, int64_t K, void *C, int out_dtype, hipStream_t st);
int launch_big_grouped(const void *Aq, const void *As, const void *Bq, const void *Bs, int scale_dtype,
                       const int32_t *m_offsets, int E, int64_t M_total, int64_t N, int64_t K, void *C, int out_dtype,
                       hipStream_t st, const int32_t *host_offsets = nullptr);

}  // namespace gemm
}  // namespace lowp
