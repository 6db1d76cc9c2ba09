// teal_rows.hip — matrix products over a few rows (a batch's step, a short prompt): y = x W^T for up to 64 rows of x, over the W^T
// images the decode step streams (row-major [K][ld], column-major weights of the host's [N, K]).  gfx950 / CDNA4, wave64; fp16, bf16.
//
// Bound by HBM: every weight byte is read once for all rows.  A workgroup owns a column tile and a slice of K; its waves take 32-row
// steps of the image in turn, two steps in flight each (teal_rows_core.h), the rows of x come as matrix-core operands straight from
// the cache (128 KB for 16 rows of 4096, read by every tile), and the waves are added in fixed order through LDS.  Split over K the
// partial sums stay in fp32 slabs [slice][row][column] for the consumer to add in slice order, or the last slice of a tile to arrive adds
// them in that order: bit-reproducible.
//
// 16 rows, bf16, us (the vendor's product): 4096 -> 4096 9.2 (15.7), 11008 -> 4096 17.0 (58), 4096 -> 10816 21 (22.5), -> 32000 42.5 (54),
// -> 2 x 11008 with the activation 38 (53 + 5), 2048 -> 2048 5.3 (9.6); 64 rows: 14.3 (22), 23 (65), 25 (28.5), 55 (50 + 4).  What is left to
// the floor (6.4 TB/s: 5.2, 14.1, 13.8, 41, 28): launch and drain, and 172 gate | up tiles on 256 CUs.
#include "teal_rows_core.h"

#include <algorithm>

namespace teal {

struct RowsArgs {
    const uint16_t* x;        // [M][ldx]
    const uint16_t* w[2];     // image [K][ld]; IM = 2: gate, up (same ld)
    const uint16_t* bias[2];  // or null: [N]
    void* y;                  // ROUNDED: 16-bit [M][ldy]; F32: fp32 [M][ldy]; SLABS: fp32 [slices][M][N]
    float* part;              // ROUNDED, F32 over several slices: partial sums [tile][slice][M][tile width * IM]
    unsigned* tickets;        // ... and a zero counter per tile, zero again afterwards
    int ldx, ld, ldy, M, K, N, act;
    int nvalid;               // F32: columns stored
    float cap;                // F32: > 0: cap * tanh(v / cap)
};

constexpr int kRowsWaves = 8, kRowsMaxRows = 64, kRowsMaxSlices = 16;

template <bool BF16>
__device__ __forceinline__ float round16(const float v) { return bits_to_float(float_to_bits<BF16>(v), BF16); }

template <bool BF16>
__device__ __forceinline__ float rows_act(const int act, const float z) {
    switch (act) {
        case TEAL_ACT_SILU: return z * sigmoid_f(z);
        case TEAL_ACT_GELU_TANH: return gelu_tanh_f(z);
        case TEAL_ACT_RELU2: return relu2_f(z);
        default: return z;
    }
}

// MT: row tiles of 16; COLS: columns per lane, a tile is 16 COLS wide; IM = 2: gate and up tiles of the same columns; OUT: TEAL_ROWS_*
template <bool BF16, int MT, int COLS, int IM, int OUT>
__global__ __launch_bounds__(64 * kRowsWaves, MT * COLS * IM <= 8 ? 4 : 2) void rows_gemm_kernel(const RowsArgs a) {
    constexpr int WAVES = kRowsWaves, F = COLS * IM, TW = 16 * COLS, LR = TW * IM + 4;  // columns per lane; tile width of an image; padded row of the reduction
    extern __shared__ __align__(16) float rows_red[];                                  // [wave][16][LR]
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, g = lane >> 4;
    const int tile = blockIdx.x, slice = blockIdx.y, split = gridDim.y, steps = a.K >> 5, ldb = 2 * a.ld;
    const int first = (int)((long long)steps * slice / split), n = (int)((long long)steps * (slice + 1) / split) - first;
    const int wide = min(TW, a.N - tile * TW);  // (the last tile may be narrower)
    RowsBuf buf[IM];
#pragma unroll
    for (int m = 0; m < IM; ++m) buf[m] = rows_buffer(a.w[m] + (size_t)tile * TW + (size_t)first * 16 * ldb, (size_t)(32 * n - 1) * ldb + 2 * wide);
    const bool mine = COLS * l16 < wide;
    const uint32_t base = (uint32_t)(8 * g) * (uint32_t)ldb + (uint32_t)(2 * COLS) * (uint32_t)l16;
    auto off = [&](const int s) { return mine && s < n ? base + (uint32_t)s * 32u * (uint32_t)ldb : kRowsNowhere; };
    const uint16_t* xp[MT];
#pragma unroll
    for (int r = 0; r < MT; ++r) xp[r] = a.x + (size_t)min(16 * r + l16, a.M - 1) * a.ldx + first * 32 + 8 * g;
    auto loadx = [&](u32x4 (&x)[MT], const int s) {
        const int at = 32 * min(s, n - 1);
#pragma unroll
        for (int r = 0; r < MT; ++r) x[r] = *reinterpret_cast<const u32x4*>(xp[r] + at);
    };
    RowsTile<COLS, IM> t0, t1;
    u32x4 x0[MT], x1[MT];
    loadx(x0, wave);
    rows_load<COLS, IM>(t0, buf, off(wave), ldb);
    loadx(x1, wave + WAVES);
    rows_load<COLS, IM>(t1, buf, off(wave + WAVES), ldb);
    f32x4 acc[MT][F];
#pragma unroll
    for (int r = 0; r < MT; ++r)
#pragma unroll
        for (int f = 0; f < F; ++f) acc[r][f] = f32x4{0.f, 0.f, 0.f, 0.f};
    int s = wave;
    for (; s + WAVES < n; s += 2 * WAVES) {
        rows_mfma<BF16, false, MT, COLS, IM>(t0, x0, acc);
        loadx(x0, s + 2 * WAVES);
        rows_load<COLS, IM>(t0, buf, off(s + 2 * WAVES), ldb);
        rows_mfma<BF16, false, MT, COLS, IM>(t1, x1, acc);
        loadx(x1, s + 3 * WAVES);
        rows_load<COLS, IM>(t1, buf, off(s + 3 * WAVES), ldb);
    }
    if (s < n) rows_mfma<BF16, false, MT, COLS, IM>(t0, x0, acc);

    constexpr int Q = TW / 4, NT = 64 * WAVES;  // quads of columns per row and image
    // the complete sums of four columns of row m
    auto emit = [&](f32x4 (&v)[IM], const int m, const int col) {
#pragma unroll
        for (int k = 0; k < IM; ++k)
            if (a.bias[k]) {
                const u32x2 b = *reinterpret_cast<const u32x2*>(a.bias[k] + col);
#pragma unroll
                for (int j = 0; j < 4; ++j) v[k][j] += bits_to_float(j & 1 ? b[j >> 1] >> 16 : b[j >> 1] & 0xFFFFu, BF16);
            }
        if constexpr (OUT == TEAL_ROWS_F32) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (col + j < a.nvalid) reinterpret_cast<float*>(a.y)[(size_t)m * a.ldy + col + j] = a.cap > 0.0f ? a.cap * tanhf(v[0][j] / a.cap) : v[0][j];
        } else {
            uint32_t o[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float z;
                if (IM == 2 && a.act == TEAL_ACT_SILU_ROUNDED) {  // (gate, up and silu(gate) each rounded to 16 bits, gpt-fast/model.py:258-259)
                    const float gt = round16<BF16>(v[0][j]);
                    z = round16<BF16>(gt / (1.0f + expf(-gt))) * round16<BF16>(v[IM - 1][j]);
                } else {
                    z = rows_act<BF16>(a.act, v[0][j]);
                    if constexpr (IM == 2) z *= v[1][j];
                }
                o[j] = float_to_bits<BF16>(z);
            }
            *reinterpret_cast<u32x2*>(reinterpret_cast<uint16_t*>(a.y) + (size_t)m * a.ldy + col) = u32x2{o[0] | (o[1] << 16), o[2] | (o[3] << 16)};
        }
    };
    float* part = OUT == TEAL_ROWS_SLABS ? nullptr : a.part + (size_t)tile * split * a.M * (TW * IM);
    // the waves in fixed order through LDS, a row tile at a time.  A lane holds row l16 and, of column group 4 g + i, the columns COLS * (4 g
    // + i) ..: 4 COLS consecutive ones per image
#pragma unroll
    for (int r = 0; r < MT; ++r) {
        if (r) __syncthreads();
        float* own = rows_red + (size_t)(wave * 16 + l16) * LR + 4 * COLS * g;
#pragma unroll
        for (int m = 0; m < IM; ++m)
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int c = 0; c < COLS; c += 4)
                    *reinterpret_cast<f32x4*>(own + m * TW + i * COLS + c) =
                        f32x4{acc[r][m * COLS + c][i], acc[r][m * COLS + c + 1][i], acc[r][m * COLS + c + 2][i], acc[r][m * COLS + c + 3][i]};
        __syncthreads();
        for (int u = tid; u < 16 * Q; u += NT) {
            const int row = u / Q, q = u % Q, m = 16 * r + row, col = tile * TW + 4 * q;
            if (m >= a.M || 4 * q >= wide) continue;
            f32x4 v[IM];
#pragma unroll
            for (int k = 0; k < IM; ++k) {
                v[k] = *reinterpret_cast<const f32x4*>(rows_red + (size_t)row * LR + k * TW + 4 * q);
#pragma unroll
                for (int w = 1; w < WAVES; ++w) v[k] += *reinterpret_cast<const f32x4*>(rows_red + (size_t)(w * 16 + row) * LR + k * TW + 4 * q);
            }
            if constexpr (OUT == TEAL_ROWS_SLABS) {
                *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(a.y) + ((size_t)slice * a.M + m) * a.N + col) = v[0];
            } else if (split == 1) {
                emit(v, m, col);
            } else {  // write-through (agent scope): another XCD's workgroup may read it
#pragma unroll
                for (int k = 0; k < IM; ++k)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        __hip_atomic_store(part + ((size_t)slice * a.M + m) * (TW * IM) + k * TW + 4 * q + j, v[k][j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
    if constexpr (OUT != TEAL_ROWS_SLABS) {
        if (split == 1) return;
        // the last slice of the tile to arrive adds the partial sums in slice order, whoever it is
        __shared__ unsigned last;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // every storing wave drains its stores
        __syncthreads();
        if (tid == 0) last = __hip_atomic_fetch_add(a.tickets + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)split - 1u;
        __syncthreads();
        if (!last) return;
        for (int u = tid; u < a.M * Q; u += NT) {
            const int m = u / Q, q = u % Q;
            if (4 * q >= wide) continue;
            f32x4 v[IM];
#pragma unroll
            for (int k = 0; k < IM; ++k) v[k] = f32x4{0.f, 0.f, 0.f, 0.f};
            for (int sl = 0; sl < split; ++sl)
#pragma unroll
                for (int k = 0; k < IM; ++k)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        v[k][j] += __hip_atomic_load(part + ((size_t)sl * a.M + m) * (TW * IM) + k * TW + 4 * q + j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            emit(v, m, tile * TW + 4 * q);
        }
        if (tid == 0) __hip_atomic_store(a.tickets + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

constexpr size_t rows_lds(const int cols, const int im) { return (size_t)kRowsWaves * 16 * (16 * cols * im + 4) * sizeof(float); }

template <bool BF16, int MT, int COLS, int IM, int OUT>
int rows_launch(const RowsArgs& a, const int split, hipStream_t st) {
    hipLaunchKernelGGL((rows_gemm_kernel<BF16, MT, COLS, IM, OUT>), dim3((a.N + 16 * COLS - 1) / (16 * COLS), split), dim3(64 * kRowsWaves), rows_lds(COLS, IM), st, a);
    return launched();
}

template <bool BF16, int MT>
int rows_mode(const RowsArgs& a, const int mode, const int split, hipStream_t st) {
    if (a.w[1]) return rows_launch<BF16, MT, 4, 2, TEAL_ROWS_ROUNDED>(a, split, st);
    if (mode == TEAL_ROWS_SLABS) return rows_launch<BF16, MT, 8, 1, TEAL_ROWS_SLABS>(a, split, st);
    if (mode == TEAL_ROWS_F32) return rows_launch<BF16, MT, 8, 1, TEAL_ROWS_F32>(a, split, st);
    return rows_launch<BF16, MT, 8, 1, TEAL_ROWS_ROUNDED>(a, split, st);
}

template <bool BF16>
int rows_tiles(const RowsArgs& a, const int mode, const int split, hipStream_t st) {
    if (a.M <= 16) return rows_mode<BF16, 1>(a, mode, split, st);
    if (a.M <= 32) return rows_mode<BF16, 2>(a, mode, split, st);
    return rows_mode<BF16, 4>(a, mode, split, st);
}

// the reductions take a few KB more than the 64 KB a kernel gets unasked (first use of a device, device_ctx())
bool rows_device_init() {
    bool ok = true;
#define TEAL_OPT1(BF, MTV, C, I, O) ok = ok && hipFuncSetAttribute(reinterpret_cast<const void*>(&rows_gemm_kernel<BF, MTV, C, I, O>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)rows_lds(C, I)) == hipSuccess
#define TEAL_OPT(BF, MTV) TEAL_OPT1(BF, MTV, 4, 2, TEAL_ROWS_ROUNDED); TEAL_OPT1(BF, MTV, 8, 1, TEAL_ROWS_SLABS); TEAL_OPT1(BF, MTV, 8, 1, TEAL_ROWS_F32); TEAL_OPT1(BF, MTV, 8, 1, TEAL_ROWS_ROUNDED)
    TEAL_OPT(false, 1); TEAL_OPT(false, 2); TEAL_OPT(false, 4); TEAL_OPT(true, 1); TEAL_OPT(true, 2); TEAL_OPT(true, 4);
#undef TEAL_OPT
#undef TEAL_OPT1
    if (!ok) (void)hipGetLastError();
    return ok;
}

// Slices of K: as many as keep the launch within one workgroup per CU (more leave a ragged second round: 4096 -> 12288, 16 rows, 192
// workgroups 20.0 us, 288 24.5), a 32-row step per wave at least
int rows_slices(const int K, const int N, const bool paired, const int ncu) {
    const int tiles = paired ? (N + 63) / 64 : (N + 127) / 128;
    return std::max(1, std::min({ncu / tiles, (K >> 5) / kRowsWaves, kRowsMaxSlices}));
}

}  // namespace teal

using namespace teal;

extern "C" {

int teal_rows_split(int M, int K, int N, int paired) {
    if (M <= 0 || K <= 0 || N <= 0) return TEAL_ERR_ARG;
    if (M > kRowsMaxRows || (K & 31) || (N & 7)) return 0;
    DeviceCtx* ctx = device_ctx();
    if (!ctx) return TEAL_ERR_NO_DEVICE;
    return ctx->rows_lds_ok ? rows_slices(K, N, paired != 0, ctx->num_cu) : 0;
}

int teal_rows_gemm(const teal_rows_gemm_t* p, int dtype, void* stream) {
    if (!p || !p->x || !p->w || !p->y || p->M <= 0 || p->K <= 0 || p->N <= 0) return TEAL_ERR_ARG;
    if (dtype != TEAL_F16 && dtype != TEAL_BF16) return TEAL_ERR_DTYPE;
    if (p->mode != TEAL_ROWS_ROUNDED && p->mode != TEAL_ROWS_SLABS && p->mode != TEAL_ROWS_F32) return TEAL_ERR_ARG;
    if ((p->w_up && p->mode != TEAL_ROWS_ROUNDED) || (p->bias_up && !p->w_up) || (p->mode != TEAL_ROWS_ROUNDED && (p->bias || p->act != TEAL_ACT_NONE))) return TEAL_ERR_ARG;
    if (p->act < TEAL_ACT_NONE || p->act > TEAL_ACT_SILU_ROUNDED || (p->act == TEAL_ACT_SILU_ROUNDED && !p->w_up)) return TEAL_ERR_ARG;
    const int split = teal_rows_split(p->M, p->K, p->N, p->w_up != nullptr);
    if (split < 0) return split;
    if (split == 0 || p->ldx < p->K || (p->ldx & 7) || p->ld < p->N || (p->ld & 7)) return TEAL_ERR_SHAPE;
    if (p->mode != TEAL_ROWS_SLABS && p->ldy < (p->mode == TEAL_ROWS_F32 ? p->n_valid : p->N)) return TEAL_ERR_SHAPE;
    if (p->mode == TEAL_ROWS_ROUNDED && (p->ldy & 3)) return TEAL_ERR_SHAPE;
    if (p->mode == TEAL_ROWS_F32 && (p->n_valid < 1 || p->n_valid > p->N)) return TEAL_ERR_SHAPE;
    if ((unsigned long long)p->K * (unsigned long long)p->ld * 2ull > 0xFFF00000ull) return TEAL_ERR_SHAPE;  // (32-bit buffer offsets)
    const void* ps[] = {p->x, p->w, p->w_up, p->bias, p->bias_up, p->part};
    for (const void* q : ps)
        if (!aligned16(q)) return TEAL_ERR_ALIGN;
    if (reinterpret_cast<uintptr_t>(p->y) & (p->mode == TEAL_ROWS_SLABS ? 15u : 7u)) return TEAL_ERR_ALIGN;
    const size_t tiled = p->w_up ? (size_t)((p->N + 63) / 64) * 128 : (size_t)((p->N + 127) / 128) * 128;
    if (p->mode != TEAL_ROWS_SLABS && split > 1 && (!p->part || !p->tickets || p->part_bytes < (size_t)split * p->M * tiled * sizeof(float))) return TEAL_ERR_WORKSPACE;
    RowsArgs a = {};
    a.x = reinterpret_cast<const uint16_t*>(p->x);
    a.w[0] = reinterpret_cast<const uint16_t*>(p->w);
    a.w[1] = reinterpret_cast<const uint16_t*>(p->w_up);
    a.bias[0] = reinterpret_cast<const uint16_t*>(p->bias);
    a.bias[1] = reinterpret_cast<const uint16_t*>(p->bias_up);
    a.y = p->y; a.part = p->part; a.tickets = p->tickets;
    a.ldx = p->ldx; a.ld = p->ld; a.ldy = p->ldy; a.M = p->M; a.K = p->K; a.N = p->N; a.act = p->act; a.nvalid = p->n_valid; a.cap = p->softcap;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    return dtype == TEAL_BF16 ? rows_tiles<true>(a, p->mode, split, st) : rows_tiles<false>(a, p->mode, split, st);
}

}  // extern "C"
