// teal_rows_core.h — the core of the matrix products over a few rows (teal_prefill.hip, teal_rows.hip): a wave streams rows of the
// W^T image the decode kernels read and multiplies them on the matrix cores.  Internal header.
//
// Bound by HBM (every weight byte is read once for all rows), so the one question is how the image's layout — a row per input
// feature, columns contiguous — becomes the matrix cores' operand, eight consecutive inputs of one column per lane.  A lane loads 16
// bytes (8 columns; 8 bytes, 4 columns) of each of eight consecutive rows: coalesced segments of 256 (128) bytes.  v_perm_b32 pairs
// the halves of two rows, and the eight rows' words ARE the operands of the lane's columns: one instruction per two weights, no LDS,
// no second copy of the weights (the vector ALU has a tenth of the stream's time to do at 6 TB/s).
#pragma once
#include "teal_prompt_attention.h"

namespace teal {

// one step of a wave: 32 rows of the image, COLS columns per lane of each of IM images; lane = (column group l & 15, row group l >> 4)
template <int COLS, int IM>
struct RowsTile {
    static_assert(COLS == 8 || COLS == 4, "16 or 8 bytes per lane and row");
    static constexpr int D = COLS / 2, F = COLS * IM;  // words per row and image; columns (operands) per lane
    uint32_t w[IM][8][D];
};

// The image as a buffer resource: a step past the last one is requested at an offset outside of it and costs nothing, so the loop
// below has no branch between its loads and its products (a branch would make the compiler wait for every load in flight)
typedef __amdgpu_buffer_rsrc_t RowsBuf;
__device__ __forceinline__ RowsBuf rows_buffer(const uint16_t* p, const size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(p), 0, (int)(uint32_t)bytes, 0x00027000);
}
constexpr uint32_t kRowsNowhere = 0xFFFFFFF0u;

// voff: byte offset of the lane's first row and column; ldb: bytes per row.  Weights are read once: non-temporal
template <int COLS, int IM>
__device__ __forceinline__ void rows_load(RowsTile<COLS, IM>& t, const RowsBuf (&b)[IM], const uint32_t voff, const int ldb) {
#pragma unroll
    for (int m = 0; m < IM; ++m)
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            if constexpr (COLS == 8) {
                const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(b[m], (int)voff, r * ldb, 2);
#pragma unroll
                for (int d = 0; d < 4; ++d) t.w[m][r][d] = v[d];
            } else {
                const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(b[m], (int)voff, r * ldb, 2);
#pragma unroll
                for (int d = 0; d < 2; ++d) t.w[m][r][d] = v[d];
            }
        }
}

// acc[mt][f]: products of row tile mt (16 rows of x) and the lane's column f of the tile.  XA: x is the first operand — acc's lane
// holds column f of group l & 15, rows 4 * (l >> 4) + i; else it holds row l & 15 and column f of the groups 4 * (l >> 4) + i
template <bool BF16, bool XA, int MT, int COLS, int IM>
__device__ __forceinline__ void rows_mfma(const RowsTile<COLS, IM>& t, const u32x4 (&x)[MT], f32x4 (&acc)[MT][COLS * IM]) {
#pragma unroll
    for (int m = 0; m < IM; ++m)
#pragma unroll
        for (int d = 0; d < COLS / 2; ++d) {
            u32x4 lo, hi;
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                lo[p] = __builtin_amdgcn_perm(t.w[m][2 * p + 1][d], t.w[m][2 * p][d], 0x05040100u);
                hi[p] = __builtin_amdgcn_perm(t.w[m][2 * p + 1][d], t.w[m][2 * p][d], 0x07060302u);
            }
            const int f = m * COLS + 2 * d;
#pragma unroll
            for (int r = 0; r < MT; ++r) {
                if constexpr (XA) {
                    acc[r][f] = mfma16<BF16>(x[r], lo, acc[r][f]);
                    acc[r][f + 1] = mfma16<BF16>(x[r], hi, acc[r][f + 1]);
                } else {
                    acc[r][f] = mfma16<BF16>(lo, x[r], acc[r][f]);
                    acc[r][f + 1] = mfma16<BF16>(hi, x[r], acc[r][f + 1]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);  // (all the permutes first would take another 32 registers)
        }
}

}  // namespace teal
