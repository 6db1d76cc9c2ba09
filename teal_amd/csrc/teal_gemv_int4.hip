// teal_gemv_int4.hip — sparse GEMV over int4 group-quantised weights.
//
// The reference ships int4-g32/64/128 weight-only linears for its DENSE gpt-fast path only
// (gpt-fast/quantize.py:58-162 group q-params / quantise / dequantise, :359-443 handler, :483-526 WeightOnlyInt4Linear,
// whose forward is a CUDA-only tinygemm op) and lists quantised TEAL as missing (README.md:110).  Semantics restated:
//     w[n][m] = (q[n][m] - 8) * scale[m / G][n] + zero[m / G][n]        q in 0..15, scale / zero bf16, G = group size
//     y[n]    = sum over kept m of x[m] * w[n][m]                        kept: float32(|x[m]|) > float32(tau), strict
// scales_and_zeros [Z / G][N][2] bf16 exactly as the reference stores them (quantize.py:79-93).
//
// Weight layout (ours to choose — the reference's packed layout is tinygemm's): the image of W^T by ROW PAIRS,
// wq[Z / 2][ldb] bytes; dword g of pair-row p holds columns 4g .. 4g+3 of row 2p in its low half (nibble j = column 4g+j)
// and of row 2p+1 in its high half.  One mask-and-or under a 16-bit exponent yields (1024 + q[2p][c], 1024 + q[2p+1][c])
// (fp16; bf16: 128 + q), two of the eight inputs of one column that a lane hands the matrix cores.  A pair is
// fetched when EITHER row is kept (the other row's x enters as 0, which is exact): at 50 % sparsity 75 % of the pairs.
//
// Kernel: one 16-wave workgroup = one 128-column tile x one slice of the 32-row units; a wave takes every sixteenth unit.  The
// workgroup leaves its slice's activations masked in LDS; a lane (8 columns, the four pairs of its 16-lane group) reads its eight
// with one LDS read, requests the pairs whose activations are not both zero (the others at an offset outside the buffer
// resource: no traffic, no list, no branch), and eight MFMAs give sum x * (bias + q) of the unit's 32 rows, a ninth, over ones,
// X = sum x.  Scale and zero are applied ONCE per (unit, column):  y += scale * (A - (bias + 8) X) + zero * X.  The 16 waves keep
// one unit each in flight.  Split-K over units is folded into the one launch by arrival tickets (the last slice of a tile sums the
// partials in slice order: deterministic, no atomics on the data).
//
// What bounds it: the vector ALU (72 instructions per unit and wave, half of them nibbles becoming halves), then the launch's fixed 4 - 5
// us; the stream (weights and, at G = 32, a quarter as many bytes of group parameters) hides behind them: with nothing kept a launch is
// only a fifth faster.  Llama-2-7B at G = 32 and 50 %: gate|up 16.8 -> 15.1, qkv 11.7 -> 10.5, down 8.6 -> 7.5, wo 7.8 -> 5.7 us.
// The kernel before this one compacted the kept pairs into lists and walked them with v_dot2, 16 dot products and 9 list
// instructions per pair and lane: bound by the vector ALU and by its passes (ballots -> lists -> loads -> products, nothing of one
// pass in flight during the next).
//
// The kernel takes the producers of the fused decode step like the 16-bit one (teal_gemv_fast.h): MODE 1 residual + fp32
// slabs -> RMSNorm (every workgroup recomputes the whole vector: the norm needs all of it), MODE 2 silu(gate) * up and
// MODE 4 split-KV attention merge (element-wise: a workgroup builds its own slice) — and leaves either rounded outputs or its
// fp32 split-K partials as slabs for the next launch's producer, so an int4 layer is 5 launches too.
#include "teal_rows_core.h"

#include <limits.h>

// Same rule as the 16-bit GEMV units (teal_gemv_kernel.h): no implicit contraction — every fused multiply-add below is an
// explicit fmaf(), so the slab path and the rounded path, and this unit against the merge producers elsewhere, cannot drift
// by an ulp when the compiler changes its mind.
#pragma clang fp contract(off)
#include <stdio.h>

namespace teal {

constexpr int kPhaseRow = 32;  // uint64 stamps per workgroup (as in teal_gemv_kernel.h)

struct I4Seg {
    const unsigned char* wq;  // first byte of the segment's columns in pair-row 0
    const uint16_t* sz;       // (scale, zero) of the segment's first column in group 0
    uint16_t* y;              // rounded output of the segment (null when the launch leaves slabs)
    int ldb, szld;            // pair-row stride of wq in bytes; columns per row of sz
    int tile0;                // first 128-column tile of the segment
    float tau;
};

struct I4Args {
    I4Seg seg[3];
    int nseg, Z, gshift;      // gshift: log2 of the group size
    // producer
    const uint16_t* x;        // MODE 0: x[Z]; MODE 2: gate[Z] | up[Z]; MODE 1: residual (table with row_index)
    const int* row_index;
    const float* slabs;       // MODE 1: interleaved fp32 partials [Z][(nslabs + 3) & ~3] folded into the residual
    int nslabs;
    const uint16_t* norm_w;
    float eps;
    uint16_t* resid_out;
    const float* att;         // MODE 4: partials [Z / hd][ns][hd + 2]
    int att_hd, att_ns;
    // split-K partials / slabs: element (column c, slice s) at ws[c * ws_es + s * ws_ss]
    float* ws;
    int ws_es, ws_ss;
    unsigned* ticket;         // null: split == 1, or the partials stay as slabs for the consumer
    unsigned long long* phase;  // PHASE instantiations: kPhaseRow stamps per workgroup (teal_set_phase_buffer)
};

// fp16 activations: nibbles 1 and 3 of a half are used where they lie, as 1024 + 16 q (no shift); their columns are rescaled when
// scale and zero are applied.  bf16 activations: bias 128 (7 mantissa bits), every nibble shifted down.
// PHASE (measurement builds only): thread 0 stamps [0] entry, [1] arguments in registers, [2] MODE 1's producer done, [3] activations in LDS,
// [5] first unit requested, [6] first unit consumed, [8] all units done, [9] past the reduce barrier, [10] outputs stored.
// 100 MHz wall clock (scripts/int4_phase.py).
constexpr size_t kI4MaxLds = 128 * 1024 + 64;  // masked activations of a slice (65536 rows) and one unit of zeros
template <bool BF16, int MODE, bool PHASE = false>
__global__ __launch_bounds__(1024) void sparse_gemv_int4_kernel(const I4Args a) {
    constexpr int WAVES = 16, BN = 128, DEPTH = 1;  // DEPTH: units of a wave in flight (2, 3, 4: 4, 7, 11 % slower per token)
    unsigned long long t_entry = 0;
    if constexpr (PHASE) t_entry = wall_clock64();
    extern __shared__ __align__(16) uint16_t xs[];  // masked activations: MODE 1 the whole vector, else the slice's units back to back
    __shared__ __align__(16) float red[WAVES * BN];
    __shared__ float wsum[WAVES];
    __shared__ float tflag;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int tile = blockIdx.x, slice = blockIdx.y, split = gridDim.y;
    const int g = lane >> 4, cl = lane & 15;  // the lane's four pairs of a unit, its 8 columns of the tile
    const int Z = a.Z;
    auto stamp = [&](const int i) {
        if constexpr (PHASE) {
            if (a.phase && tid == 0) a.phase[(size_t)(blockIdx.y * gridDim.x + blockIdx.x) * kPhaseRow + i] = wall_clock64();
        }
    };
    // ONE batch of scalar loads for every kernel argument, up front (an "s" input forces the value into an SGPR here):
    // left to the compiler they are fetched where first used — a chain of dependent scalar-cache misses through the
    // prologue and again in the epilogue
#define TEAL_I4_SEG_ARGS(g) "s"((g).wq), "s"((g).sz), "s"((g).y), "s"((g).ldb), "s"((g).szld), "s"((g).tile0), "s"((g).tau)
    asm volatile("" ::TEAL_I4_SEG_ARGS(a.seg[0]), TEAL_I4_SEG_ARGS(a.seg[1]), TEAL_I4_SEG_ARGS(a.seg[2]));
    asm volatile("" ::"s"(a.nseg), "s"(a.Z), "s"(a.gshift), "s"(a.x), "s"(a.row_index), "s"(a.slabs), "s"(a.nslabs), "s"(a.norm_w),
                 "s"(a.eps), "s"(a.resid_out), "s"(a.att), "s"(a.att_hd), "s"(a.att_ns), "s"(a.ws), "s"(a.ws_es), "s"(a.ws_ss),
                 "s"(a.ticket));
#undef TEAL_I4_SEG_ARGS
    if constexpr (PHASE) {
        if (a.phase && tid == 0) a.phase[(size_t)(blockIdx.y * gridDim.x + blockIdx.x) * kPhaseRow] = t_entry;
    }
    stamp(1);

    // ---- this workgroup's column tile: segment, threshold, weight image ---------------------------------------------------
    // (selected field by field from kernel arguments already in SGPRs: indexing a.seg[] by a run-time s would be a
    // dependent scalar load)
    int s = 0;
    if (a.nseg > 1 && tile >= a.seg[1].tile0) s = 1;
    if (a.nseg > 2 && tile >= a.seg[2].tile0) s = 2;
#define TEAL_I4_SEG(f) (s == 0 ? a.seg[0].f : (s == 1 ? a.seg[1].f : a.seg[2].f))
    const unsigned char* seg_wq = TEAL_I4_SEG(wq);
    const uint16_t* seg_sz = TEAL_I4_SEG(sz);
    uint16_t* seg_y = TEAL_I4_SEG(y);
    const int ldb = TEAL_I4_SEG(ldb), szld = TEAL_I4_SEG(szld), seg_tile0 = TEAL_I4_SEG(tile0);
    const float tau = TEAL_I4_SEG(tau);
#undef TEAL_I4_SEG
    auto masked = [&](const uint32_t b) -> uint16_t {
        const float v = bits_to_float(b, BF16);
        return keep_rule(v, tau) || v != v ? (uint16_t)b : (uint16_t)0;
    };
    // unit u belongs to slice u % split, and inside the slice, as its k-th, to wave k % 16
    const int nunits = Z >> 5, nk = (nunits - slice + split - 1) / split;
    // ---- producer -------------------------------------------------------------------------------------------------------
    if constexpr (MODE == 1) {
        // h = resid + round(sum slabs);  x = round(round(h * rstd) * w)          gpt-fast/model.py:158-161, 289-291
        // KM elements per thread (4: Z <= 4096, 8: Z <= 8192, else 16); every load is unconditional (index clamped) and
        // leaves in one batch (KM = 16: per block of 4 elements)
        const uint16_t* resid = a.x;
        if (a.row_index) resid += (size_t)a.row_index[0] * (size_t)Z;  // embedding row of the current token
        const uint32_t stride = (uint32_t)(a.nslabs + 3) & ~3u;
        const int nslabs = a.nslabs;
        const bool writer = a.resid_out && tile == 0 && slice == 0;
        auto produce = [&](auto km_tag) {
            constexpr int KM = decltype(km_tag)::value, KB = KM <= 8 ? KM : 4;
            uint32_t wb[KM];
#pragma unroll
            for (int k = 0; k < KM; ++k) wb[k] = a.norm_w[min(tid + (k << 10), Z - 1)];
            float ss = 0.0f;
#pragma unroll
            for (int k0 = 0; k0 < KM; k0 += KB) {
                uint32_t rb[KB];
                f32x4 v0[KB], v1[KB];
#pragma unroll
                for (int j = 0; j < KB; ++j) {
                    const uint32_t m = (uint32_t)min(tid + ((k0 + j) << 10), Z - 1);
                    rb[j] = resid[m];
                    if (nslabs > 0) v0[j] = *reinterpret_cast<const f32x4*>(a.slabs + m * stride);
                    if (nslabs > 4) v1[j] = *reinterpret_cast<const f32x4*>(a.slabs + m * stride + 4);
                }
#pragma unroll
                for (int j = 0; j < KB; ++j) {
                    const int m = tid + ((k0 + j) << 10);
                    float r = bits_to_float(rb[j], BF16);
                    if (nslabs > 0) {  // slab order 0, 1, 2, ... (the order of the ordered reduce); an absent slab adds 0.0f
                        float sacc = 0.0f;
#pragma unroll
                        for (int q = 0; q < 4; ++q) sacc += (q < nslabs) ? v0[j][q] : 0.0f;
                        if (nslabs > 4) {
#pragma unroll
                            for (int q = 0; q < 4; ++q) sacc += (4 + q < nslabs) ? v1[j][q] : 0.0f;
                        }
                        const float yv = bits_to_float(float_to_bits<BF16>(sacc), BF16);
                        r = bits_to_float(float_to_bits<BF16>(r + yv), BF16);
                    }
                    if (m < Z) {
                        xs[m] = float_to_bits<BF16>(r);  // exact: r is a 16-bit value
                        ss = fmaf(r, r, ss);
                    }
                }
            }
            ss = wave_sum_f(ss);
            if (lane == 0) wsum[wave] = ss;
            __syncthreads();
            float tot = lane < WAVES ? wsum[lane] : 0.0f;
            tot = wave_sum_f(tot);
            const float rstd = rsqrtf(tot / (float)Z + a.eps);
#pragma unroll
            for (int k = 0; k < KM; ++k) {
                const int m = tid + (k << 10);
                if (m < Z) {
                    const uint32_t hb = xs[m];  // this thread's own element
                    const float xn = bits_to_float(float_to_bits<BF16>(bits_to_float(hb, BF16) * rstd), BF16);
                    xs[m] = masked(float_to_bits<BF16>(xn * bits_to_float(wb[k], BF16)));
                    if (writer) a.resid_out[m] = (uint16_t)hb;
                }
            }
        };
        if (Z <= 4096) produce(std::integral_constant<int, 4>{});
        else if (Z <= 8192) produce(std::integral_constant<int, 8>{});
        else produce(std::integral_constant<int, 16>{});
        if (tid < 32) xs[Z + tid] = 0;
        __syncthreads();
    }

    stamp(2);
    // the element-wise producers: the slice's elements, every load of a round first
    if constexpr (MODE != 1) {
        constexpr int R = MODE == 4 ? 2 : 4;
        const int total = nk * 32;
        for (int e0 = tid; e0 < total; e0 += 1024 * R) {
            uint32_t m_el[R], xb[R];
#pragma unroll
            for (int i = 0; i < R; ++i) {
                const int e = min(e0 + 1024 * i, total - 1);
                m_el[i] = ((uint32_t)(slice + split * (e >> 5)) << 5) + (uint32_t)(e & 31);
            }
            if constexpr (MODE == 0) {
#pragma unroll
                for (int i = 0; i < R; ++i) xb[i] = a.x[m_el[i]];
            } else if constexpr (MODE == 2) {
                // x = round(round(silu(gate)) * up)                                  gpt-fast/model.py:258-259
                uint32_t gb[R], ub[R];
#pragma unroll
                for (int i = 0; i < R; ++i) {
                    gb[i] = a.x[m_el[i]];
                    ub[i] = a.x[(uint32_t)Z + m_el[i]];
                }
#pragma unroll
                for (int i = 0; i < R; ++i) {
                    const float gt = bits_to_float(gb[i], BF16);
                    const float sl = bits_to_float(float_to_bits<BF16>(gt / (1.0f + expf(-gt))), BF16);
                    xb[i] = float_to_bits<BF16>(sl * bits_to_float(ub[i], BF16));
                }
            } else {
                // attention output merged from the split-KV partials {max, sum, o[hd]} per (head, split); the arithmetic of the
                // 16-bit kernel's merge producer: pairwise-tree sum of the rescaled denominators, fmaf chain over the splits
                const int hd = a.att_hd, hs = hd + 2;
                auto merge = [&](auto ns_tag) {
                    constexpr int NS = decltype(ns_tag)::value;
                    float2 st[R][NS];
                    float ov[R][NS];
#pragma unroll
                    for (int j = 0; j < R; ++j) {
                        const int m = (int)m_el[j];
                        const int h = m / hd, d = m - h * hd;
                        const float* b = a.att + (size_t)h * NS * hs;
#pragma unroll
                        for (int q = 0; q < NS; ++q) {
                            st[j][q] = *reinterpret_cast<const float2*>(b + q * hs);
                            ov[j][q] = b[q * hs + 2 + d];
                        }
                    }
#pragma unroll
                    for (int j = 0; j < R; ++j) {
                        float M = st[j][0].x;
#pragma unroll
                        for (int q = 1; q < NS; ++q) M = fmaxf(M, st[j][q].x);
                        float f[NS], t[NS];
#pragma unroll
                        for (int q = 0; q < NS; ++q) {
                            f[q] = st[j][q].y > 0.0f ? expf(st[j][q].x - M) : 0.0f;
                            t[q] = st[j][q].y * f[q];
                        }
                        float Ls = (t[0] + t[1]) + (t[2] + t[3]);
                        if constexpr (NS == 8) Ls = Ls + ((t[7] + t[6]) + (t[5] + t[4]));
                        float Os = 0.0f;
#pragma unroll
                        for (int q = 0; q < NS; ++q) Os = fmaf(ov[j][q], f[q] / Ls, Os);
                        xb[j] = float_to_bits<BF16>(Os);
                    }
                };
                if (a.att_ns == 8) merge(std::integral_constant<int, 8>{});
                else merge(std::integral_constant<int, 4>{});
            }
#pragma unroll
            for (int i = 0; i < R; ++i)
                if (e0 + 1024 * i < total) xs[e0 + 1024 * i] = masked(xb[i]);
        }
        if (tid < 32) xs[total + tid] = 0;
        __syncthreads();
    }
    stamp(3);
    // ---- the stream ----------------------------------------------------------------------------------------------------------
    const uint32_t uldb = (uint32_t)ldb, col = (uint32_t)(tile - seg_tile0) * BN;
    const RowsBuf wbuf = rows_buffer(reinterpret_cast<const uint16_t*>(seg_wq + col), (size_t)(Z / 2 - 1) * ldb + BN);
    const RowsBuf pbuf = rows_buffer(seg_sz + 2 * (size_t)col, (size_t)((Z >> a.gshift) - 1) * szld * 4 + BN * 4);
    constexpr uint32_t kBias = BF16 ? 0x43004300u : 0x64006400u;  // (128, 128) bf16 / (1024, 1024) fp16
    constexpr uint32_t kOnes = BF16 ? 0x3F803F80u : 0x3C003C00u;  // (1, 1)
    struct Unit {
        u32x4 x;     // the lane's eight masked activations (rows 8 g ..)
        u32x2 w[4];  // its four pairs
        u32x2 p;     // (scale, zero) of columns 8 cl + 2 g and the next
    } st[DEPTH];
    // (units past the last read the zeros behind the activations, so nothing is requested for them; no branch: the loads in flight are counted)
    const int xpast = MODE == 1 ? Z : nk * 32;
    auto read_x = [&](const int k) {
        const int at = MODE == 1 ? (slice + split * k) << 5 : k << 5;
        return *reinterpret_cast<const u32x4*>(xs + (k < nk ? at : xpast) + 8 * g);
    };
    uint32_t loff[4];  // the lane's pair i inside a unit
#pragma unroll
    for (int i = 0; i < 4; ++i) loff[i] = (uint32_t)(4 * g + i) * uldb + 8u * (uint32_t)cl;
    const uint32_t poff = 32u * (uint32_t)cl + 8u * (uint32_t)g;
    auto request = [&](Unit& t, const int k) {
        const int u = slice + split * min(k, nk - 1);
        t.x = read_x(k);
#pragma unroll
        for (int i = 0; i < 4; ++i) t.w[i] = __builtin_amdgcn_raw_buffer_load_b64(wbuf, (int)(t.x[i] ? loff[i] : kRowsNowhere), (int)((uint32_t)u * 16u * uldb), 2);
        t.p = __builtin_amdgcn_raw_buffer_load_b64(pbuf, (int)poff, (int)(((uint32_t)(u << 5) >> a.gshift) * (uint32_t)szld * 4u), 0);
    };
    u32x4 ones = {kOnes, kOnes, kOnes, kOnes};
    uint32_t bias = kBias;
    asm volatile("" : "+v"(ones), "+v"(bias));  // (kept in registers: with a literal the mask-and-or would be two instructions)
    // Lane group g finishes columns 2 g, 2 g + 1 of the lane's eight, so the product of column j is wanted in the rows 4 (j / 2) .. of the
    // result only: the first operand is x in the lanes of those rows and zeros in the others — read from the zeros behind the
    // activations —, and the even and the odd columns each add up in one accumulator, no selection afterwards
    const int bank = cl >> 2;
    float total0 = 0.0f, total1 = 0.0f;
    auto consume = [&](const Unit& t, const int k) {
        const int at = MODE == 1 ? (slice + split * k) << 5 : k << 5;
        f32x4 even = {0.f, 0.f, 0.f, 0.f}, odd = even;
        u32x4 xb[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) xb[q] = *reinterpret_cast<const u32x4*>(xs + (bank == q ? at : xpast) + 8 * g);
        const float X = mfma16<BF16>(t.x, ones, even)[0];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int h = q >> 1;
            u32x4 be, bo;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t w = t.w[i][h];
                if constexpr (BF16) {
                    be[i] = ((q & 1 ? w >> 8 : w) & 0x000F000Fu) | bias;
                    bo[i] = ((q & 1 ? w >> 12 : w >> 4) & 0x000F000Fu) | bias;
                } else {
                    const uint32_t v = q & 1 ? w >> 8 : w;
                    be[i] = (v & 0x000F000Fu) | bias;
                    bo[i] = (v & 0x00F000F0u) | bias;  // 1024 + 16 q
                }
            }
            even = mfma16<BF16>(xb[q], be, even);
            odd = mfma16<BF16>(xb[q], bo, odd);
        }
        const float s0 = __uint_as_float(t.p[0] << 16), z0 = __uint_as_float(t.p[0] & 0xFFFF0000u), s1 = __uint_as_float(t.p[1] << 16), z1 = __uint_as_float(t.p[1] & 0xFFFF0000u);
        // sum x (q - 8) from the biased sums
        const float t0 = fmaf(BF16 ? -136.0f : -1032.0f, X, even[0]), t1 = BF16 ? fmaf(-136.0f, X, odd[0]) : fmaf(odd[0], 0.0625f, -72.0f * X);
        total0 += fmaf(s0, t0, z0 * X);
        total1 += fmaf(s1, t1, z1 * X);
    };
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) request(st[i], wave + WAVES * i);
    stamp(5);
    int k = wave;
    for (; k + WAVES * (DEPTH - 1) < nk; k += WAVES * DEPTH) {
#pragma unroll
        for (int i = 0; i < DEPTH; ++i) {
            consume(st[i], k + WAVES * i);
            __builtin_amdgcn_sched_barrier(0);
            request(st[i], k + WAVES * (DEPTH + i));
        }
        if (k == wave) stamp(6);
    }
#pragma unroll
    for (int i = 0; i < DEPTH - 1; ++i)
        if (k + WAVES * i < nk) consume(st[i], k + WAVES * i);
    stamp(8);
    // ---- reduce: the waves in fixed order ------------------------------------------------------------------------------------
    *reinterpret_cast<float2*>(red + wave * BN + 8 * cl + 2 * g) = make_float2(total0, total1);
    __syncthreads();
    stamp(9);
    const uint32_t c = (uint32_t)tile * BN + tid;  // column in the concatenation of the segments (slab / partial index)
    uint16_t* yp = seg_y ? seg_y + (uint32_t)(tile - seg_tile0) * BN + tid : nullptr;
    float sum = 0.0f;
    if (tid < BN) {
#pragma unroll
        for (int w = 0; w < WAVES; ++w) sum += red[w * BN + tid];
        if (!a.ws) *yp = float_to_bits<BF16>(sum);
        else if (a.ticket) __hip_atomic_store(&a.ws[c * (uint32_t)a.ws_es + (uint32_t)slice * a.ws_ss], sum, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else a.ws[c * (uint32_t)a.ws_es + (uint32_t)slice * a.ws_ss] = sum;  // slabs for the next launch's producer
    }
    if (a.ticket) {  // arrival tickets: see gemv_fast_kernel
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0) {
            const unsigned t = __hip_atomic_fetch_add(&a.ticket[tile], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            tflag = (t == (unsigned)split - 1u) ? 1.0f : 0.0f;
        }
        __syncthreads();
        if (tflag != 0.0f && tid < BN) {
            float acc = 0.0f;
            for (int sl = 0; sl < split; ++sl)
                acc += __hip_atomic_load(&a.ws[c * (uint32_t)a.ws_es + (uint32_t)sl * a.ws_ss], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            *yp = float_to_bits<BF16>(acc);
            if (tid == 0) __hip_atomic_store(&a.ticket[tile], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if constexpr (PHASE) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        stamp(10);
    }
}

template <bool BF16, bool PHASE>
static hipError_t launch_i4(const I4Args& a, int mode, dim3 grid, size_t lds, hipStream_t st) {
    const dim3 block(1024);
    switch (mode) {
        case TEAL_IN_PLAIN: hipLaunchKernelGGL((sparse_gemv_int4_kernel<BF16, 0, PHASE>), grid, block, lds, st, a); break;
        case TEAL_IN_RESID_NORM: hipLaunchKernelGGL((sparse_gemv_int4_kernel<BF16, 1, PHASE>), grid, block, lds, st, a); break;
        case TEAL_IN_SILU_MUL: hipLaunchKernelGGL((sparse_gemv_int4_kernel<BF16, 2, PHASE>), grid, block, lds, st, a); break;
        default: hipLaunchKernelGGL((sparse_gemv_int4_kernel<BF16, 4, PHASE>), grid, block, lds, st, a); break;
    }
    return hipGetLastError();
}

// vectors beyond 28672 rows a slice need more LDS than a kernel gets unasked (first use of a device, device_ctx())
bool int4_device_init() {
    bool ok = true;
#define TEAL_OPT(BF, M) ok = ok && hipFuncSetAttribute(reinterpret_cast<const void*>(&sparse_gemv_int4_kernel<BF, M>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)kI4MaxLds) == hipSuccess
    TEAL_OPT(false, 0); TEAL_OPT(false, 1); TEAL_OPT(false, 2); TEAL_OPT(false, 4); TEAL_OPT(true, 0); TEAL_OPT(true, 1); TEAL_OPT(true, 2); TEAL_OPT(true, 4);
#undef TEAL_OPT
    if (!ok) (void)hipGetLastError();
    return ok;
}

// One launch over int4 weights: [producer] -> mask + compaction -> gathered GEMV over every segment (teal_fused_gemv with
// weight_bits = 4, and the plain entry point below).  split-K factor: enough slices to cover the CUs, at most 8, every
// wave of every slice owning at least one unit; without a destination for the partials (no prepared workspace and no
// slabs requested) the launch keeps every unit of a tile in one workgroup.
int fused_gemv_i4(const teal_gemv_in_t* in, const teal_gemv_out_t* out, int Z, int dtype, void* ws, size_t ws_bytes,
                  int* nslabs_out, hipStream_t st) {
    const int G = out->groupsize;
    if (G != 32 && G != 64 && G != 128 && G != 256) return TEAL_ERR_ARG;
    if (Z <= 0 || (Z % G) || Z > 65536) return TEAL_ERR_SHAPE;
    if (out->nseg < 1 || out->nseg > 3) return TEAL_ERR_ARG;
    if (out->mode != TEAL_OUT_ROUNDED && out->mode != TEAL_OUT_SLABS) return TEAL_ERR_ARG;  // no paired gate|up form
    DeviceCtx* dc = device_ctx();
    if (!dc) return TEAL_ERR_NO_DEVICE;
    I4Args a = {};
    a.nseg = out->nseg; a.Z = Z; a.gshift = G == 32 ? 5 : (G == 64 ? 6 : (G == 128 ? 7 : 8));
    int ntiles = 0, N = 0;
    for (int i = 0; i < out->nseg; ++i) {
        const int nc = out->ncols[i], c0 = out->col0[i], ldb = out->ld[i], szld = out->scale_ld[i];
        if (!out->w[i] || !out->scale[i] || nc <= 0 || (nc % 128) || c0 < 0 || (c0 & 7)) return TEAL_ERR_SHAPE;
        if (ldb < c0 + nc || (ldb & 7) || szld < c0 + nc) return TEAL_ERR_SHAPE;  // a pair-row: one byte per column
        if ((size_t)(Z / 2) * (size_t)ldb >= ((size_t)1 << 32)) return TEAL_ERR_SHAPE;  // 32-bit offsets inside an image
        if ((reinterpret_cast<uintptr_t>(out->w[i]) & 7u) || !aligned16(out->scale[i])) return TEAL_ERR_ALIGN;
        if (out->mode == TEAL_OUT_ROUNDED && !out->y[i]) return TEAL_ERR_ARG;
        I4Seg& sg = a.seg[i];
        sg.wq = reinterpret_cast<const unsigned char*>(out->w[i]) + c0;
        sg.sz = reinterpret_cast<const uint16_t*>(out->scale[i]) + (size_t)c0 * 2;
        sg.y = out->mode == TEAL_OUT_ROUNDED ? reinterpret_cast<uint16_t*>(out->y[i]) : nullptr;
        sg.ldb = ldb; sg.szld = szld; sg.tile0 = ntiles; sg.tau = out->tau[i];
        ntiles += nc / 128;
        N += nc;
    }
    size_t lds = 0;
    switch (in->mode) {
        case TEAL_IN_PLAIN:
            if (!in->x) return TEAL_ERR_ARG;
            a.x = reinterpret_cast<const uint16_t*>(in->x);
            break;
        case TEAL_IN_SILU_MUL:
            if (!in->x) return TEAL_ERR_ARG;
            a.x = reinterpret_cast<const uint16_t*>(in->x);
            break;
        case TEAL_IN_ATTN_MERGE:
            if (!in->x || (in->att_head_dim != 64 && in->att_head_dim != 128) || Z % in->att_head_dim ||
                (in->att_nsplit != 0 && in->att_nsplit != 4 && in->att_nsplit != 8))
                return TEAL_ERR_ARG;
            a.att = reinterpret_cast<const float*>(in->x);
            a.att_hd = in->att_head_dim;
            a.att_ns = in->att_nsplit ? in->att_nsplit : 4;
            break;
        case TEAL_IN_RESID_NORM:
            if (!in->resid_in || !in->norm_weight || in->nslabs < 0 || (in->nslabs > 0 && !in->slabs)) return TEAL_ERR_ARG;
            if (in->resid_out == in->resid_in && !in->row_index) return TEAL_ERR_ARG;  // must ping-pong
            if (in->nslabs > 0 && (!in->slabs_interleaved || in->nslabs > 8 || !aligned16(in->slabs))) return TEAL_ERR_ARG;
            if (Z > 16384) return TEAL_ERR_SHAPE;  // 16 elements per thread, 32 KB of LDS
            a.x = reinterpret_cast<const uint16_t*>(in->resid_in);
            a.row_index = in->row_index;
            a.slabs = in->slabs;
            a.nslabs = in->nslabs;
            a.norm_w = reinterpret_cast<const uint16_t*>(in->norm_weight);
            a.eps = in->eps;
            a.resid_out = reinterpret_cast<uint16_t*>(in->resid_out);
            lds = (size_t)Z * 2 + 64;
            break;
        default: return TEAL_ERR_ARG;  // TEAL_IN_MASKED: no int4 form
    }
    const int nunits = Z / 32;
    int split = dc->num_cu / ntiles;
    if (split > 8) split = 8;
    if (split * 16 > nunits) split = nunits / 16;  // every wave of every slice owns at least one 32-row unit
    if (split < 1) split = 1;
    if (out->mode == TEAL_OUT_SLABS) {
        if (!out->slabs || !aligned16(out->slabs) || ws_prepared(out->slabs, out->slabs_bytes)) return TEAL_ERR_ARG;
        a.ws = out->slabs;
        if (out->slabs_interleaved) { a.ws_es = (split + 3) & ~3; a.ws_ss = 1; }
        else { a.ws_es = 1; a.ws_ss = N; }
        if (out->slabs_bytes < (size_t)(out->slabs_interleaved ? a.ws_es : split) * N * sizeof(float)) return TEAL_ERR_WORKSPACE;
    } else if (split > 1) {
        if (!ws_prepared(ws, ws_bytes) || ntiles > kTicketTiles) split = 1;
        else {
            a.ws_es = (split + 3) & ~3; a.ws_ss = 1;
            if (ws_bytes - kWsHeaderBytes < (size_t)a.ws_es * N * sizeof(float)) return TEAL_ERR_WORKSPACE;
            a.ws = ws_slabs(ws);
            a.ticket = ws_tickets(ws);
        }
    }
    const dim3 grid(ntiles, split);
    if (in->mode != TEAL_IN_RESID_NORM) lds = (size_t)((nunits + split - 1) / split) * 64 + 64;
    if (lds > 56 * 1024 && !dc->int4_lds_ok) return TEAL_ERR_LAUNCH;
    hipError_t e;
#ifdef TEAL_DIAGNOSTICS
    if (g_phase && dtype == TEAL_F16) {  // measurement: the stamping instantiation (fp16 only; libteal_hip_diag.so)
        a.phase = phase_next_region();
        e = launch_i4<false, true>(a, in->mode, grid, lds, st);
    } else
#endif
    if (dtype == TEAL_BF16) {
        e = launch_i4<true, false>(a, in->mode, grid, lds, st);
    } else {
        e = launch_i4<false, false>(a, in->mode, grid, lds, st);
    }
    if (e != hipSuccess) return TEAL_ERR_LAUNCH;
    if (out->desc || kDiagnostics) {
        char d[160];
        snprintf(d, sizeof d, "sparse_gemv_int4_kernel<%s,%d,false> grid (%d,%d) x 1024", dtype == TEAL_BF16 ? "true" : "false",
                 in->mode, ntiles, split);
        publish_desc(d, out->desc, out->desc_bytes);
    }
    if (nslabs_out) *nslabs_out = split;
    return TEAL_OK;
}

}  // namespace teal

using namespace teal;

extern "C" int teal_sparse_qkv_gemv_i4(const void* x, const void* wq, const void* scales_and_zeros, void* y, float tau_q,
                                       float tau_k, float tau_v, int Z, int N, int N_q, int N_kv, int ldb, int groupsize,
                                       int dtype, void* ws, size_t ws_bytes, void* stream) {
    if (!x || !wq || !scales_and_zeros || !y || Z <= 0 || N <= 0) return TEAL_ERR_ARG;
    if (dtype != TEAL_F16 && dtype != TEAL_BF16) return TEAL_ERR_DTYPE;
    if (groupsize != 32 && groupsize != 64 && groupsize != 128 && groupsize != 256) return TEAL_ERR_ARG;
    if ((N % 128) || (Z % groupsize) || Z > 65536 || ldb < N || (ldb & 7)) return TEAL_ERR_SHAPE;
    if (N_q <= 0 || N_kv < 0 || N_q + 2 * N_kv != N || (N_q % 128) || (N_kv % 128)) return TEAL_ERR_SHAPE;
    teal_gemv_in_t in = {};
    in.mode = TEAL_IN_PLAIN;
    in.x = x;
    teal_gemv_out_t out = {};
    out.nseg = N_kv > 0 ? 3 : 1;
    const int c0[3] = {0, N_q, N_q + N_kv}, nc[3] = {N_q, N_kv, N_kv};
    const float tau[3] = {tau_q, tau_k, tau_v};
    for (int i = 0; i < out.nseg; ++i) {
        out.w[i] = wq; out.scale[i] = scales_and_zeros;
        out.ld[i] = ldb; out.scale_ld[i] = N;
        out.col0[i] = c0[i]; out.ncols[i] = nc[i]; out.tau[i] = tau[i];
        out.y[i] = reinterpret_cast<uint16_t*>(y) + c0[i];
    }
    out.mode = TEAL_OUT_ROUNDED;
    out.weight_bits = 4;
    out.groupsize = groupsize;
    return fused_gemv_i4(&in, &out, Z, dtype, ws, ws_bytes, nullptr, reinterpret_cast<hipStream_t>(stream));
}
