// Row-scaled FP8 GEMM for problems of one K block (gemm_rowscale_small) and of two (gemm_rowscale_strip): the weight
// gradients dW_e = dY_e^T X_e of experts with at most 256 rows (gpatch_v4/models/deepseek_v4/fp8.py:325-341), which are most
// experts of a routed batch.  Such a problem is a write of M x N results more than a GEMM: a 128 x 128 tile reads 32 KB (or
// 64 KB) and writes 32 KB of bf16.  With one K block there is no pipeline inside a workgroup: it requests its whole operand
// tiles (LDS-direct loads, 8 rows x 128 bytes per request), waits once, multiplies with the scale bytes of both operands
// applied by the matrix cores, stages the results through the same LDS and stores whole 128-byte lines.  What overlaps one
// workgroup's wait and stores is the other workgroups of its CU: 36 KB of LDS and 64 accumulators per lane let four of them
// share it.  LDS rows and chunks are laid out as in gemm_fp8_big.hip (the 16 lanes of a fragment read cover whole 256-byte
// lines).
//
// Two K blocks leave room for two workgroups only, too few to cover each other's wait for 64 KB: that way 15 problems of
// 4096 x 4096 took 159 us, 3.2 TB/s of results, where the strips take 114 (bound by their stores: 40 problems of 7168 x 4096
// reach 5.4 TB/s).  gemm_rowscale_strip keeps a workgroup's activation rows in registers and walks a strip of weight columns, the
// next tile's operand on its way while this one is multiplied and stored.
#include "gemm_common.h"

using namespace lowp;

namespace {

typedef int i32x8 __attribute__((ext_vector_type(8)));
typedef float f32x4v __attribute__((ext_vector_type(4)));

#define LDS_PTR(p) ((void __attribute__((address_space(3))) *)(p))
#define GLB_PTR(p) ((const void __attribute__((address_space(1))) *)(p))

// LDS row that holds tile row r, the tile row an LDS row holds, and the slot of chunk c of tile row r
__device__ __forceinline__ int lds_row(int r) { return (r & ~15) | ((r & 7) << 1) | ((r >> 3) & 1); }
__device__ __forceinline__ int tile_row(int p) { return (p & ~15) | ((p >> 1) & 7) | ((p & 1) << 3); }
__device__ __forceinline__ int swz(int r, int chunk) { return chunk ^ (r & 7); }

// bf16 results of a wave's 64 x 64 sub-tile through LDS: row pitch 128 + 16 bytes, written per accumulator block (mb, nb)
// by lane (l16, lq) -- row 16 mb + l16, columns 16 nb + 4 lq .. + 3 -- and read back in 16-byte chunks of 8 columns, 8
// lanes to a row, so that a store instruction writes 8 whole rows of 128 bytes.
constexpr int kPitch = 64 * 2 + 16, kWaveStage = 64 * kPitch;

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 4))) void gemm_rowscale_small(
    const uint8_t *__restrict__ Aq, const uint8_t *__restrict__ As, const uint8_t *__restrict__ Bq, const uint8_t *__restrict__ Bs,
    const int32_t *__restrict__ groups, int G, int64_t M, int64_t N, uint32_t tiles_m, uint32_t tiles_n, int shift, void *__restrict__ C,
    int out_dtype)
{
    constexpr int TILE = 128 * 128, PITCH = 128;
    __shared__ __attribute__((aligned(1024))) uint8_t smem[2 * TILE > 4 * kWaveStage ? 2 * TILE : 4 * kWaveStage];
    int64_t g, tm, tn;
    if (!gemm::list_coords(blockIdx.x, (uint32_t)G, tiles_m, tiles_n, shift, g, tm, tn)) return;
    // no table: one problem
    const int64_t slot = groups ? groups[4 * g] : 0, kb = groups ? groups[4 * g + 1] : 1, before = groups ? groups[4 * g + 2] : 0;
    // an entry of another size (or one that breaks the caller's promises) is not this launch's: nothing is written
    if (kb != 1 || slot < 0 || before < 0) return;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wave >> 1, wn = wave & 1, l16 = lane & 15, lq = lane >> 4;
    const int64_t m0 = tm * 128, n0 = tn * 128;
    const uint8_t *a_g = Aq + M * 128 * before + m0 * PITCH, *b_g = Bq + N * 128 * before + n0 * PITCH;
    const uint8_t *as_g = As + M * before + m0, *bs_g = Bs + N * before + n0;

    // requests: group q of 8 LDS rows of an operand block is wave q % 4's; lane -> row lane / 8 of the group, slot lane % 8
    const int ld_row = lane >> 3, ld_slot = lane & 7;
    uint32_t off[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = tile_row(8 * (wave + 4 * i) + ld_row);
        off[i] = (uint32_t)(row * PITCH + swz(row, ld_slot) * 16);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int q = wave + 4 * i;
        __builtin_amdgcn_global_load_lds(GLB_PTR(a_g + off[i]), LDS_PTR(smem + q * 1024), 16, 0, 0);
        __builtin_amdgcn_global_load_lds(GLB_PTR(b_g + off[i]), LDS_PTR(smem + TILE + q * 1024), 16, 0, 0);
    }
    int sa[4], sb[4];                                    // scale bytes of the lane's rows
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        sa[b] = as_g[wm * 64 + b * 16 + l16];
        sb[b] = bs_g[wn * 64 + b * 16 + l16];
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();

    f32x4v acc[4][4];
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) acc[mb][nb] = f32x4v{0.0f, 0.0f, 0.0f, 0.0f};
    auto frag = [&](const uint8_t *base, int row) -> i32x8 {
        const u32x4 x0 = *(const u32x4 *)(base + lds_row(row) * 128 + swz(row, 2 * lq) * 16);
        const u32x4 x1 = *(const u32x4 *)(base + lds_row(row) * 128 + swz(row, 2 * lq + 1) * 16);
        return i32x8{(int)x0.x, (int)x0.y, (int)x0.z, (int)x0.w, (int)x1.x, (int)x1.y, (int)x1.z, (int)x1.w};
    };
    // fragments are read where they are used (the activation side four times over): registers for four workgroups per CU
#pragma unroll
    for (int nb = 0; nb < 4; ++nb) {
        const i32x8 bf = frag(smem + TILE, wn * 64 + nb * 16 + l16);
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) {
            const i32x8 af = frag(smem, wm * 64 + mb * 16 + l16);
            acc[mb][nb] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(bf, af, acc[mb][nb], 0, 0, 0, sb[nb], 0, sa[mb]);
        }
    }

    const int64_t row0 = m0 + wm * 64, col0 = n0 + wn * 64;
    char *c_g = (char *)C + slot * M * N * (out_dtype == LP_BF16 ? 2 : 4);
    if (out_dtype == LP_BF16) {
        __syncthreads();                                 // every wave has read its fragments: the tile memory is free
        uint8_t *stage = smem + wave * kWaveStage;
#pragma unroll
        for (int mb = 0; mb < 4; ++mb)
#pragma unroll
            for (int nb = 0; nb < 4; ++nb) {
                const u32x2 o = {pack_bf16(acc[mb][nb].x, acc[mb][nb].y), pack_bf16(acc[mb][nb].z, acc[mb][nb].w)};
                *(u32x2 *)(stage + (mb * 16 + l16) * kPitch + (nb * 16 + 4 * lq) * 2) = o;
            }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // a wave reads back only what it wrote
#pragma unroll
        for (int p = 0; p < 8; ++p) {
            const int row = p * 8 + (lane >> 3), chunk = lane & 7;
            const u32x4 v = *(const u32x4 *)(stage + row * kPitch + chunk * 16);
            __builtin_nontemporal_store(v, (u32x4 *)((uint16_t *)c_g + (row0 + row) * N + col0 + chunk * 8));
        }
        return;
    }
#pragma unroll
    for (int mb = 0; mb < 4; ++mb)
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
            const u32x4 o = {f2u(acc[mb][nb].x), f2u(acc[mb][nb].y), f2u(acc[mb][nb].z), f2u(acc[mb][nb].w)};
            *(u32x4 *)((float *)c_g + (row0 + mb * 16 + l16) * N + col0 + nb * 16 + 4 * lq) = o;
        }
}

// Problems of two K blocks: a 128-row panel of A against `strip` 128-column tiles of B, one after the other.  The panel's
// fragments stay in registers (64 of them); B tiles go through two 32 KB halves of LDS, tile i + 1 requested before tile i is
// multiplied.  When a tile's fragments have been read its half takes the bf16 results (64 x 64 per wave, 128-byte rows,
// 16-byte chunks swizzled so that neither side has bank conflicts) on their way to whole-line stores.  The wait for the next
// tile stands in front of those stores (loads and stores share the request counter, and stores acknowledge late).
constexpr int kStripTile = 128 * 128, kStripHalf = 2 * kStripTile;

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void gemm_rowscale_strip(
    const uint8_t *__restrict__ Aq, const uint8_t *__restrict__ As, const uint8_t *__restrict__ Bq, const uint8_t *__restrict__ Bs,
    const int32_t *__restrict__ groups, int G, int64_t M, int64_t N, int tiles_m, int tiles_n, int strip, int piece, void *__restrict__ C, int out_dtype)
{
    __shared__ __attribute__((aligned(1024))) uint8_t smem[2 * kStripHalf];
    // The strips of all problems are numbered problem by problem and strip by strip, row panels running fastest, and pieces of
    // `piece` consecutive ones, which share a strip of B in an L2, are dealt to the XCDs (workgroup id modulo 8) in turn.
    const int runs = tiles_m * ((tiles_n + strip - 1) / strip), in_xcd = blockIdx.x >> 3;
    const int id = (in_xcd / piece * 8 + (blockIdx.x & 7)) * piece + in_xcd % piece, g = id / runs, run = id - g * runs;
    if (g >= G) return;
    const int first_n = run / tiles_m * strip, tm = run % tiles_m;
    const int count = tiles_n - first_n < strip ? tiles_n - first_n : strip;
    // no table: one problem.  An entry of another size (or one that breaks the caller's promises) is not this launch's:
    // nothing is written
    const int64_t slot = groups ? groups[4 * g] : 0, kb = groups ? groups[4 * g + 1] : 2, before = groups ? groups[4 * g + 2] : 0;
    if (kb != 2 || slot < 0 || before < 0) return;
    const int t = threadIdx.x, lane = t & 63;
    const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const int wm = wave >> 1, wn = wave & 1, l16 = lane & 15, lq = lane >> 4;
    const int64_t m0 = (int64_t)tm * 128, n0 = (int64_t)first_n * 128;
    const uint8_t *a_g = Aq + M * 128 * before + m0 * 256, *b_g = Bq + N * 128 * before + n0 * 256;
    const uint8_t *as_g = As + M * before + m0 * 2, *bs_g = Bs + N * before + n0 * 2;

    // requests as in gemm_rowscale_small: group q of 8 LDS rows of a K block is wave q % 4's
    uint32_t off[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int row = tile_row(8 * (wave + 4 * i) + (lane >> 3));
        off[i] = (uint32_t)(row * 256 + swz(row, lane & 7) * 16);
    }
    const uint32_t lds0 = (uint32_t)(uintptr_t)LDS_PTR(smem) + (uint32_t)wave * 1024;
    // (not the builtin: behind it the compiler waits for the request in front of every LDS read)
    auto request = [&](const uint8_t *tile, int half) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                             :: "s"(lds0 + (uint32_t)(half * kStripHalf + j * kStripTile + i * 4096)), "v"(off[i]), "s"(tile + j * 128)
                             : "memory", "m0");
    };
    auto frag = [&](const uint8_t *base, int row) -> i32x8 {
        const u32x4 x0 = *(const u32x4 *)(base + lds_row(row) * 128 + swz(row, 2 * lq) * 16);
        const u32x4 x1 = *(const u32x4 *)(base + lds_row(row) * 128 + swz(row, 2 * lq + 1) * 16);
        return i32x8{(int)x0.x, (int)x0.y, (int)x0.z, (int)x0.w, (int)x1.x, (int)x1.y, (int)x1.z, (int)x1.w};
    };
    request(a_g, 1);
    request(b_g, 0);
    // scale bytes of the lane's rows: byte j of the register = K block j (picked by the instruction's op_sel)
    int sa[4], sb[4];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        sa[b] = *(const uint16_t *)(as_g + 2 * (wm * 64 + b * 16 + l16));
        sb[b] = *(const uint16_t *)(bs_g + 2 * (wn * 64 + b * 16 + l16));
    }
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" : "+v"(sa[0]), "+v"(sa[1]), "+v"(sa[2]), "+v"(sa[3]), "+v"(sb[0]), "+v"(sb[1]), "+v"(sb[2]), "+v"(sb[3]) :: "memory");
    i32x8 af[2][4];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int mb = 0; mb < 4; ++mb) af[j][mb] = frag(smem + kStripHalf + j * kStripTile, wm * 64 + mb * 16 + l16);
    const int64_t esz = out_dtype == LP_BF16 ? 2 : 4;
    char *c_g = (char *)C + (slot * M * N + (m0 + wm * 64) * N + n0 + wn * 64) * esz;
    for (int i = 0; i < count; ++i) {
        // every wave is through with the other half (the A panel, or the results of the tile before), and this tile has landed
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        uint8_t *half = smem + (i & 1) * kStripHalf;
        const bool more = i + 1 < count;
        int sn[4] = {0, 0, 0, 0};
        if (more) {
            request(b_g + (int64_t)(i + 1) * (128 * 256), (i + 1) & 1);
#pragma unroll
            for (int b = 0; b < 4; ++b) sn[b] = *(const uint16_t *)(bs_g + (int64_t)(i + 1) * 256 + 2 * (wn * 64 + b * 16 + l16));
        }
        f32x4v acc[4][4];
#pragma unroll
        for (int mb = 0; mb < 4; ++mb)
#pragma unroll
            for (int nb = 0; nb < 4; ++nb) acc[mb][nb] = f32x4v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int nb = 0; nb < 4; ++nb) {
            const i32x8 b0 = frag(half, wn * 64 + nb * 16 + l16), b1 = frag(half + kStripTile, wn * 64 + nb * 16 + l16);
#pragma unroll
            for (int mb = 0; mb < 4; ++mb)
                acc[mb][nb] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(b0, af[0][mb], acc[mb][nb], 0, 0, 0, sb[nb], 0, sa[mb]);
#pragma unroll
            for (int mb = 0; mb < 4; ++mb)
                acc[mb][nb] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(b1, af[1][mb], acc[mb][nb], 0, 0, 1, sb[nb], 1, sa[mb]);
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");      // every wave has read this tile's fragments
        if (out_dtype == LP_BF16) {
            uint8_t *stage = half + wave * (64 * 128);
#pragma unroll
            for (int mb = 0; mb < 4; ++mb)
#pragma unroll
                for (int nb = 0; nb < 4; ++nb) {
                    const u32x2 o = {pack_bf16(acc[mb][nb].x, acc[mb][nb].y), pack_bf16(acc[mb][nb].z, acc[mb][nb].w)};
                    const int row = mb * 16 + l16, chunk = nb * 2 + (lq >> 1);
                    *(u32x2 *)(stage + row * 128 + (chunk ^ ((row >> 1) & 7)) * 16 + (lq & 1) * 8) = o;
                }
        }
        // the next tile has landed (and the stores of the tile before are done); a wave reads back only what it wrote
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" : "+v"(sn[0]), "+v"(sn[1]), "+v"(sn[2]), "+v"(sn[3]) :: "memory");
#pragma unroll
        for (int b = 0; b < 4; ++b) sb[b] = sn[b];
        char *c_t = c_g + (int64_t)i * 128 * esz;
        if (out_dtype == LP_BF16) {
            const uint8_t *stage = half + wave * (64 * 128);
#pragma unroll
            for (int p = 0; p < 8; ++p) {
                const int row = p * 8 + (lane >> 3), chunk = lane & 7;
                const u32x4 v = *(const u32x4 *)(stage + row * 128 + (chunk ^ ((row >> 1) & 7)) * 16);
                __builtin_nontemporal_store(v, (u32x4 *)((uint16_t *)c_t + (int64_t)row * N + chunk * 8));
            }
        } else {
#pragma unroll
            for (int mb = 0; mb < 4; ++mb)
#pragma unroll
                for (int nb = 0; nb < 4; ++nb) {
                    const u32x4 o = {f2u(acc[mb][nb].x), f2u(acc[mb][nb].y), f2u(acc[mb][nb].z), f2u(acc[mb][nb].w)};
                    *(u32x4 *)((float *)c_t + (int64_t)(mb * 16 + l16) * N + nb * 16 + 4 * lq) = o;
                }
        }
    }
}

}  // namespace

namespace lowp {
namespace gemm {

// Every entry of `groups` has k_blocks K blocks (1 or 2): e8m0 scales, M and N multiples of 128.  groups == nullptr: one
// problem (G = 1) written at C.
int launch_rowscale_small(const void *Aq, const void *As, const void *Bq, const void *Bs, const int32_t *groups, int G, int k_blocks,
                          int64_t M, int64_t N, void *C, int out_dtype, hipStream_t st)
{
    const int64_t tiles_m = M / 128, tiles_n = N / 128;
    if (k_blocks == 2) {
        // Strips of at most 8 tiles, all alike, cut so that rounds of two workgroups per CU x (their tiles + 2 for the panel's load and the
        // first tile's wait) are fewest: 8 tiles for many problems (40 x 7168 x 4096, strips of 2 / 4 / 8 / 16 tiles: 535 / 476 / 433 / 471 us; 15 x
        // 4096 x 4096: 117 / 122 / 114 / 128), down to one for few (one problem of 1024 x 1024 / 2048 x 2048 / 7168 x 2048, strips of 8: 14.2 us
        // each, as cut here 4.6 / 5.6 / 9.7; 8 problems of 1024 x 1024 13.9 / 6.9), and dealt out in smaller pieces until every XCD has
        // one (384 x 384 in a piece of 8 7.1, in pieces of one 4.4; below ten tiles a workgroup without a strip's two barriers more would be
        // 0.2 us ahead).
        int64_t strip = 1, best = INT64_MAX;
        for (int64_t s = 1; s <= 8 && s <= tiles_n; ++s) {
            const int64_t per_row = (tiles_n + s - 1) / s;
            if ((tiles_n + per_row - 1) / per_row != s) continue;              // not alike: a shorter strip makes as many
            const int64_t cost = (G * tiles_m * per_row + 511) / 512 * (s + 2);
            if (cost <= best) best = cost, strip = s;
        }
        const int64_t runs = G * tiles_m * ((tiles_n + strip - 1) / strip);
        int piece = GROUP_M;
        while (piece > 1 && (runs + piece - 1) / piece < 8) piece /= 2;
        const int64_t wgs = (runs + 8 * piece - 1) / (8 * piece) * (8 * piece);
        if (wgs > 0x7FFFFFFF || tiles_n > 0x7FFFFF || tiles_m > 0x7FFFFF) return fail(LP_ERR_UNSUPPORTED, "lp_gemm_fp8_rowscale_grouped: problem too large");
        hipLaunchKernelGGL(gemm_rowscale_strip, dim3((unsigned)wgs), dim3(256), 0, st, (const uint8_t *)Aq, (const uint8_t *)As, (const uint8_t *)Bq,
                           (const uint8_t *)Bs, groups, G, M, N, (int)tiles_m, (int)tiles_n, (int)strip, piece, C, out_dtype);
        return check_launch("lp_gemm_fp8_rowscale_grouped(two K blocks)");
    }
    const int shift = list_shift(G, tiles_m, tiles_n);
    const int64_t grid = list_grid(G, tiles_m, tiles_n, shift);
    if (grid > 0x7FFFFFFF) return fail(LP_ERR_UNSUPPORTED, "lp_gemm_fp8_rowscale_grouped: problem too large");
    hipLaunchKernelGGL(gemm_rowscale_small, dim3((unsigned)grid), dim3(256), 0, st, (const uint8_t *)Aq, (const uint8_t *)As, (const uint8_t *)Bq,
                       (const uint8_t *)Bs, groups, G, M, N, (uint32_t)tiles_m, (uint32_t)tiles_n, shift, C, out_dtype);
    return check_launch("lp_gemm_fp8_rowscale_grouped(one K block)");
}

}  // namespace gemm
}  // namespace lowp
