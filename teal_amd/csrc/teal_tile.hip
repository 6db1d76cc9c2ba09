// teal_tile.hip — matrix products y = x W^T of a prompt's rows over the W^T images (row-major [K][ld]).  gfx950 / CDNA4, wave64; fp16, bf16.
#include "teal_rows_core.h"

#include <algorithm>

namespace teal {

struct TileArgs {
    const uint16_t* x;     // [M][ldx]
    const uint16_t* w[2];  // images (same ld, N columns each); two: the column tiles of the second follow those of the first
    void* y[2];            // 16-bit [M][ldy], or (slabs) fp32 [slices][M][N]
    int ldx, ld, ldy, M, K, N, rows, rts, tiles, images;  // rows of a row tile (16 MT), row tiles; column tiles of one image
};

constexpr int kTileCols = 256, kTileK = 64;

// A workgroup makes 16 MT rows (48 to 160) x 256 columns, each of its four waves all the rows of 64 columns, in steps of 64 inputs.  Bound: from 65 to
// some hundred rows the image's bytes are still most of the work (11008 x 4096: 14 us), so the image goes from memory straight to the registers of
// the one wave that multiplies it, two steps ahead, is read once per row tile and by row tiles on one XCD; x, read by all four waves, goes through
// two LDS buffers.  The library's products of these sizes run with few workgroups where K is long (301 x 11008 -> 4096: 94 us; here, in eight
// slices, 46 us, and 49 with the reader's share).  More rows a wave would need more than the 256 accumulators that two waves a SIMD leave; with
// __syncthreads(), which waits for the loads in flight too, 301 rows ran at 439 TFLOP/s instead of 670.

template <bool BF16, int MT, bool SLABS>
__global__ __launch_bounds__(256, 2) void tile_gemm_kernel(const TileArgs a) {
    constexpr int BM = 16 * MT, NX = (BM * kTileK * 2 + 4095) / 4096;  // 16-byte pieces of x per thread and iteration
    __shared__ __align__(16) u32x4 xs[2][BM * kTileK / 8];             // [row tile][k step][group][row]: an operand is 1 KB on end
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, g = lane >> 4;
    // workgroup i runs on XCD i % 8: the row tiles of a column tile follow each other on one XCD, whose L2 then reads the image once
    const int at8 = blockIdx.x >> 3, rt = at8 % a.rts, ctile = (at8 / a.rts) * 8 + (blockIdx.x & 7), slice = blockIdx.y, split = gridDim.y;
    const int im = ctile >= a.tiles ? 1 : 0, ct = ctile - (im ? a.tiles : 0);
    if (ctile >= a.tiles * a.images) return;
    const int iters = a.K / kTileK, first = (int)((long long)iters * slice / split), n = (int)((long long)iters * (slice + 1) / split) - first;
    const int m0 = rt * BM, col0 = ct * kTileCols + 64 * wave, ldb = 2 * a.ld, wide = min(64, a.N - col0);
    const uint16_t* w = im ? a.w[1] : a.w[0];
    const RowsBuf buf[1] = {rows_buffer(w + (size_t)first * kTileK * a.ld + (wide > 0 ? col0 : 0), (size_t)(kTileK * n - 1) * ldb + 2 * max(wide, 4))};
    const bool mine = 4 * l16 < wide;
    const uint32_t base = (uint32_t)(8 * g) * (uint32_t)ldb + 8u * (uint32_t)l16;
    auto off = [&](const int s) { return mine && s < 2 * n ? base + (uint32_t)s * 32u * (uint32_t)ldb : kRowsNowhere; };  // (s: 32-row steps)
    // x: a thread's piece i is row tid / 8 + 32 i, inputs 8 (tid % 8) ..; rows past the last lie outside the buffer and read as zeros
    const RowsBuf xbuf = rows_buffer(a.x + (size_t)first * kTileK, ((size_t)(a.M - 1) * a.ldx + (size_t)n * kTileK) * 2);
    const int xrow = tid >> 3, xc = tid & 7;
    const uint32_t xoff = (uint32_t)(m0 + xrow) * (uint32_t)(2 * a.ldx) + 16u * (uint32_t)xc, xstep = 64u * (uint32_t)a.ldx;
    const int xat = (((xrow >> 4) * 2 + (xc >> 2)) * 4 + (xc & 3)) * 16 + ((xrow & 15) ^ xc);  // (turned by the piece: a wave's stores do not share banks)
    u32x4 xr[NX];
    auto fetch = [&](const int it) {
#pragma unroll
        for (int i = 0; i < NX; ++i) {
            const uint32_t row = (uint32_t)(m0 + xrow + 32 * i);
            xr[i] = __builtin_amdgcn_raw_buffer_load_b128(xbuf, (int)(row < (uint32_t)a.M && it < n ? xoff + i * xstep : kRowsNowhere), it < n ? it * kTileK * 2 : 0, 0);
        }
    };
    auto stash = [&](const int b) {
#pragma unroll
        for (int i = 0; i < NX; ++i)
            if (BM % 32 == 0 || xrow + 32 * i < BM) xs[b][xat + 256 * i] = xr[i];
    };
    RowsTile<4, 1> t[2];
    fetch(0);
#pragma unroll
    for (int s = 0; s < 2; ++s) rows_load<4, 1>(t[s], buf, off(s), ldb);
    f32x4 acc[MT][4];
#pragma unroll
    for (int r = 0; r < MT; ++r)
#pragma unroll
        for (int f = 0; f < 4; ++f) acc[r][f] = f32x4{0.f, 0.f, 0.f, 0.f};
    stash(0);
    for (int it = 0; it < n; ++it) {
        // (not __syncthreads(), which would wait for the loads in flight as well)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const u32x4* xb = xs[it & 1];
        fetch(it + 1);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            u32x4 b[4];
#pragma unroll
            for (int d = 0; d < 2; ++d)
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    b[2 * d][p] = __builtin_amdgcn_perm(t[s].w[0][2 * p + 1][d], t[s].w[0][2 * p][d], 0x05040100u);
                    b[2 * d + 1][p] = __builtin_amdgcn_perm(t[s].w[0][2 * p + 1][d], t[s].w[0][2 * p][d], 0x07060302u);
                }
            rows_load<4, 1>(t[s], buf, off(2 * (it + 1) + s), ldb);
#pragma unroll
            for (int r = 0; r < MT; ++r) {
                const u32x4 x = xb[((r * 2 + s) * 4 + g) * 16 + (l16 ^ (4 * s + g))];
#pragma unroll
                for (int f = 0; f < 4; ++f) acc[r][f] = mfma16<BF16>(b[f], x, acc[r][f]);
            }
        }
        stash((it + 1) & 1);
    }
    // a lane holds row l16 of each row tile and the columns 16 g .. 16 g + 15 of the wave's 64
    const int col = col0 + 16 * g;
    if (col >= a.N) return;
#pragma unroll
    for (int r = 0; r < MT; ++r) {
        const int m = m0 + 16 * r + l16;
        if (m >= a.M) continue;
        if constexpr (SLABS) {
            float* y = reinterpret_cast<float*>(a.y[0]) + ((size_t)slice * a.M + m) * a.N + col;
#pragma unroll
            for (int i = 0; i < 4; ++i) *reinterpret_cast<f32x4*>(y + 4 * i) = f32x4{acc[r][0][i], acc[r][1][i], acc[r][2][i], acc[r][3][i]};
        } else {
            uint16_t* y = reinterpret_cast<uint16_t*>(im ? a.y[1] : a.y[0]) + (size_t)m * a.ldy + col;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                u32x4 o;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    o[j] = (uint32_t)float_to_bits<BF16>(acc[r][2 * (j & 1)][2 * h + (j >> 1)]) | ((uint32_t)float_to_bits<BF16>(acc[r][2 * (j & 1) + 1][2 * h + (j >> 1)]) << 16);
                *reinterpret_cast<u32x4*>(y + 8 * h) = o;
            }
        }
    }
}

template <bool BF16, bool SLABS>
int tile_launch(const TileArgs& a, const int split, hipStream_t st) {
    const dim3 grid((a.tiles * a.images + 7) / 8 * 8 * a.rts, split);
#define TEAL_TG(MT) case 16 * MT: hipLaunchKernelGGL((tile_gemm_kernel<BF16, MT, SLABS>), grid, dim3(256), 0, st, a); return launched()
    switch (a.rows) {
        TEAL_TG(3); TEAL_TG(4); TEAL_TG(5); TEAL_TG(6); TEAL_TG(7); TEAL_TG(8); TEAL_TG(9); TEAL_TG(10);
        default: return TEAL_ERR_SHAPE;
    }
#undef TEAL_TG
}

struct TilePlan { int rows, split; };
// Rows of a tile and slices of K with the least expected time, from what launches took: a workgroup alone on its CU 36 + 0.28 rows us per 4096
// inputs (the rows share the image's loads), each further one on the same CU 0.9 of that, and partial sums written and read at 3.5 TB/s
TilePlan tile_plan(const int M, const int K, const int N, const int images, const bool slabs, const int ncu) {
    TilePlan best = {0, 1};
    float least = 1e30f;
    const int tiles = (N + kTileCols - 1) / kTileCols * images;
    for (int rows = 48; rows <= 160; rows += 16) {
        const int rts = (M + rows - 1) / rows;
        if (rows > 48 && rts == (M + rows - 17) / (rows - 16)) continue;  // (a smaller tile gives as many)
        for (int split = 1; split == 1 || (slabs && split <= 8 && split * 4 * kTileK <= K); ++split) {
            const int per_cu = (tiles * rts * split + ncu - 1) / ncu;
            const float t = (36.0f + 0.28f * rows) * (K / 4096.0f) / split * (1.0f + 0.9f * (per_cu - 1)) + (slabs ? split * (float)M * N * 8.0f / 3.5e6f : 0.0f);
            if (t < least) { least = t; best = {rows, split}; }
        }
    }
    return best;
}

}  // namespace teal

using namespace teal;

extern "C" {

int teal_tile_split(int M, int K, int N, int images, int slabs) {
    if (M <= 0 || K <= 0 || N <= 0 || images < 1 || images > 2 || (slabs && images > 1)) return TEAL_ERR_ARG;
    if ((K % kTileK) || (N & 15)) return 0;
    DeviceCtx* ctx = device_ctx();
    if (!ctx) return TEAL_ERR_NO_DEVICE;
    const TilePlan plan = tile_plan(M, K, N, images, slabs != 0, ctx->num_cu);
    // Where the library's product is the slower one (bf16, library / this kernel, with the norm that reads the result).  Partial sums: an image
    // longer than wide, which the library does not split: up to 4096 columns 11008 -> 4096 1.17 to 2.5 at 65 to 640 rows, 16384 -> 4096 1.3 to 2.8,
    // 8192 -> 2048 1.1 to 1.5, 5632 -> 2048 1.0 to 1.3; wider ones, whose column tiles leave the CUs unevenly filled, up to 160 rows (13824 -> 5120 1.07 to
    // 1.5, 320 rows 1.08, 640 0.83; 28672 -> 8192 1.25 to 2.0, 384 rows 0.89).  Square images are the library's (4096: 96 rows 30 us / 27, 256: 29 / 33; 5120: 96 rows
    // 34 / 41).  Gate and up apart (two calls of the library): from about a hundred rows on while one round of workgroups holds them
    // all (4096 -> 2 x 11008: 80 rows 0.98, 128 to 320 1.23 to 1.36, 384, a second round, 0.97; 2048 -> 2 x 5632 1.2 to 1.65; 8192 -> 2 x 28672: 160 rows 1.21, 192 0.82);
    // as one image the library has them in one call, which is faster (0.7 to 1.0)
    if (slabs ? K < 2 * N || M > (N <= 4096 ? 640 : 160)
              : images == 1 || N < 4096 || M <= 96 || M > 384 || (N + kTileCols - 1) / kTileCols * 2 * ((M + plan.rows - 1) / plan.rows) > ctx->num_cu)
        return 0;
    return plan.split;
}

int teal_tile_gemm(const void* x, int ldx, const void* w0, const void* w1, int ld, void* y0, void* y1, int ldy, float* slabs, int M, int K, int N, int dtype, void* stream) {
    if (!x || !w0 || (!w1) != (!y1) || (!y0) == (!slabs) || (slabs && w1) || M <= 0 || K <= 0 || N <= 0) return TEAL_ERR_ARG;
    if (dtype != TEAL_F16 && dtype != TEAL_BF16) return TEAL_ERR_DTYPE;
    if ((K % kTileK) || (N & 15) || ldx < K || (ldx & 7) || ld < N || (ld & 7) || (!slabs && (ldy < N || (ldy & 7)))) return TEAL_ERR_SHAPE;
    if ((unsigned long long)K * (unsigned long long)ld * 2ull > 0xFFF00000ull || (unsigned long long)M * (unsigned long long)ldx * 2ull > 0xFFF00000ull) return TEAL_ERR_SHAPE;  // (32-bit buffer offsets)
    const void* ps[] = {x, w0, w1, y0, y1, slabs};
    for (const void* p : ps)
        if (!aligned16(p)) return TEAL_ERR_ALIGN;
    DeviceCtx* ctx = device_ctx();
    if (!ctx) return TEAL_ERR_NO_DEVICE;
    const TilePlan plan = tile_plan(M, K, N, w1 ? 2 : 1, slabs != nullptr, ctx->num_cu);
    TileArgs a = {};
    a.x = reinterpret_cast<const uint16_t*>(x);
    a.w[0] = reinterpret_cast<const uint16_t*>(w0);
    a.w[1] = reinterpret_cast<const uint16_t*>(w1);
    a.y[0] = slabs ? slabs : y0;
    a.y[1] = y1;
    a.ldx = ldx; a.ld = ld; a.ldy = ldy; a.M = M; a.K = K; a.N = N;
    a.rows = plan.rows; a.rts = (M + plan.rows - 1) / plan.rows; a.tiles = (N + kTileCols - 1) / kTileCols; a.images = w1 ? 2 : 1;
    if ((long long)(a.tiles * a.images + 7) / 8 * 8 * a.rts > 0x7FFFFFFFll) return TEAL_ERR_SHAPE;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (dtype == TEAL_BF16) return slabs ? tile_launch<true, true>(a, plan.split, st) : tile_launch<true, false>(a, plan.split, st);
    return slabs ? tile_launch<false, true>(a, plan.split, st) : tile_launch<false, false>(a, plan.split, st);
}

}  // extern "C"
