// teal_prompt_attention.h — flash attention of a prompt's portions over packed keys and values, on the matrix cores (16-bit elements):
// latent attention's expanded form and grouped-query attention.  The launchers are instantiated in teal_latent.hip (scores as they
// are) and teal_prompt_attention_capped.hip (soft-capped scores).  Internal header.
#pragma once
#include "teal_layered.h"

namespace teal {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
constexpr float kLog2e = 1.4426950408889634f;
template <bool BF16>
__device__ __forceinline__ f32x4 mfma16(const u32x4 a, const u32x4 b, const f32x4 c) {
    if constexpr (BF16) return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
}

typedef short s16x4 __attribute__((ext_vector_type(4)));
// ds_read_b64_tr_b16: of 16 lanes, lane i names the 8 bytes of row i / 4, columns 4 (i % 4) of a 4 x 16 block and receives column i
__device__ __forceinline__ u32x2 lds_column4(const uint16_t* p) {
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    return __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)p));
}

// 2^x of a non-positive x (v_exp_f32: one ulp; results below the normal range are zero)
__device__ __forceinline__ float exp2_fast(const float x) { return __builtin_amdgcn_exp2f(x); }

// cap * tanh(z / cap) in log2 units: x = 2 log2(e) z / cap in, cl2 = cap * log2(e).  1 - 2 / (1 + 2^x): absolute error of an ulp of cl2
__device__ __forceinline__ float soft_cap2(const float x, const float cl2) {
    return fmaf(-2.0f * cl2, __builtin_amdgcn_rcpf(1.0f + exp2_fast(x)), cl2);
}
// the factor in front of the product that makes soft_cap2's x (capped) or a score in log2 units
template <bool CAPPED>
__device__ __forceinline__ float score_factor(const float scale, const float cap) { return CAPPED ? 2.0f * kLog2e * scale / cap : scale * kLog2e; }

// two values as packed high and low 16-bit halves
template <bool BF16>
__device__ __forceinline__ void split16x2(const float a, const float b, uint32_t& hi, uint32_t& lo) {
    if constexpr (BF16) {
        typedef float f32v2 __attribute__((ext_vector_type(2)));
        typedef __bf16 bf16v2 __attribute__((ext_vector_type(2)));
        hi = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32v2{a, b}), bf16v2));
        lo = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32v2{a - __uint_as_float(hi << 16), b - __uint_as_float(hi & 0xFFFF0000u)}), bf16v2));
    } else {
        const uint32_t h0 = float_to_bits<false>(a), h1 = float_to_bits<false>(b);
        hi = h0 | (h1 << 16);
        lo = (uint32_t)float_to_bits<false>(a - bits_to_float(h0, false)) | ((uint32_t)float_to_bits<false>(b - bits_to_float(h1, false)) << 16);
    }
}

// v as a high and a low 16-bit half
template <bool BF16>
__device__ __forceinline__ void split16(const float v, uint32_t& hi, uint32_t& lo) {
    hi = float_to_bits<BF16>(v);
    lo = float_to_bits<BF16>(v - bits_to_float(hi, BF16));
}

// ------------------------------------------------------------------------------------------------
// Flash attention over the expanded keys.
// ------------------------------------------------------------------------------------------------
struct SeqSpan {      // one sequence of the pass (five int32)
    int q0, nq;       // its rows among the packed tokens
    int start;        // position of its first row
    int k0, klo;      // packed key row of position klo (a multiple of 8), the first position packed
};

struct PromptAttentionArgs {
    const void* q;      // [T][ldq], heads x (dim + rot), rotated
    const void* k;      // [S][heads / group * dim]
    const void* kr;     // [S][rot]
    const void* vt;     // [heads / group * vdim][S]
    const void* sink;   // or null: [heads]
    const void* gate;   // or null: [T][ldg], heads x vdim
    void* out;          // [T][ldo]
    const SeqSpan* seqs;
    const int32_t* tiles;  // [ntiles][2]: sequence, first query of the tile
    int ldq, ldg, ldo, heads, group, dim, rot, vdim, S, window;
    float scale, softcap;  // softcap > 0: scores become softcap * tanh(score / softcap)
};

// S^T = K Q^T per tile: a lane then holds four consecutive keys of ONE query, which is the layout the second product's operand
// needs when the keys of two 16-key tiles are interleaved per lane group — the weights never cross lanes.  O^T = V^T P^T.
// CAP: scores as they are; capped; capped and BOUNDED — a cap of at most kBoundedCap lets 2^score stand as it is (fp32 and bf16 reach
// 2^127): no running maximum, nothing is rescaled.
constexpr float kStaleMax = 8.0f;  // a running maximum is replaced only by scores that exceed it by this much (log2 units): weights up to 2^8 meanwhile
enum { kCapNone = 0, kCapped = 1, kCapBounded = 2 };
constexpr float kBoundedCap = 60.0f;  // 2^(60 log2(e)) = 2^86.6 per key

// VEC: head sizes and row strides in whole 16 bytes.  Loads are unconditional then, at addresses clamped into the arrays, and what lies outside a head becomes
// zero on the way to the LDS: under a condition a load is followed by the copy of its result, which waits for it on the spot.
template <bool BF16, int DQP, int DVP, int NQ, int BN, int NT, int CAP, bool VEC>
__global__ __launch_bounds__(NT) void prompt_attention_kernel(const PromptAttentionArgs a) {
    constexpr int KS = DQP / 32, KT = BN / 16, VT = DVP / 16, LK = DQP + 8, LV = BN + 8, BM = NT / 4 * NQ;
    __shared__ __align__(16) uint16_t ks[BN * LK];
    __shared__ __align__(16) uint16_t vs[DVP * LV];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, g = lane >> 4;
    const int tile = blockIdx.x / a.heads, head = blockIdx.x - tile * a.heads;  // (the heads of a tile start together: the tiles come longest first)
    const SeqSpan sq = a.seqs[a.tiles[2 * tile]];
    const int q_first = a.tiles[2 * tile + 1];
    const int dq = a.dim + a.rot;
    const uint16_t* kp = reinterpret_cast<const uint16_t*>(a.k);
    const uint16_t* krp = reinterpret_cast<const uint16_t*>(a.kr);
    const int kvh = head / a.group, kvs = a.heads / a.group * a.dim;  // key / value head; row stride of the keys
    const uint16_t* vp = reinterpret_cast<const uint16_t*>(a.vt) + (size_t)kvh * a.vdim * a.S;

    u32x4 qf[NQ][KS];
    int qpos[NQ];
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        const int qi = q_first + (wave * NQ + n) * 16 + l16;
        qpos[n] = qi < sq.nq ? sq.start + qi : -1;
        const uint16_t* src = reinterpret_cast<const uint16_t*>(a.q) + (size_t)(sq.q0 + min(qi, sq.nq - 1)) * a.ldq + head * dq;
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            const int d0 = s * 32 + g * 8;
            u32x4 w = {0u, 0u, 0u, 0u};
            if constexpr (VEC) {
                if (d0 < dq) w = *reinterpret_cast<const u32x4*>(src + d0);
            } else {
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if (d0 + j < dq) w[j >> 1] |= (uint32_t)src[d0 + j] << (16 * (j & 1));
            }
            qf[n][s] = w;
        }
    }
    float m[NQ], l[NQ];
    f32x4 o[NQ][VT];
    const float sink2 = a.sink ? bits_to_float(reinterpret_cast<const uint16_t*>(a.sink)[head], BF16) * kLog2e : -INFINITY;
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        m[n] = CAP == kCapBounded ? 0.0f : sink2;
        l[n] = 0.0f;
#pragma unroll
        for (int v = 0; v < VT; ++v) o[n][v] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const int last = sq.start + min(q_first + BM, sq.nq) - 1;           // position of the tile's last query
    const int first = max(sq.klo, sq.start + q_first - a.window + 1);   // first position any of its queries sees
    const float sc = score_factor<CAP != kCapNone>(a.scale, a.softcap), cl2 = a.softcap * kLog2e;
    // the next tile's keys and values are requested while a tile is worked on
    constexpr int CK = DQP / 8, CV = BN / 8, NK = BN * CK / NT, NV = DVP * CV / NT;
    u32x4 kreg[NK], vreg[NV];
    auto fetch = [&](const int kt) {
#pragma unroll
        for (int i = 0; i < NK; ++i) {
            const int at = tid + NT * i, key = at / CK, d0 = (at % CK) * 8;
            const size_t row = (size_t)min(sq.k0 + kt + key, a.S - 1);
            if constexpr (VEC) {
                const int d = min(d0, dq - 8);
                kreg[i] = *reinterpret_cast<const u32x4*>(d < a.dim ? kp + row * kvs + kvh * a.dim + d : krp + row * a.rot + d - a.dim);
            } else {
                kreg[i] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int d = d0 + j;
                    if (d < dq) kreg[i][j >> 1] |= (uint32_t)(d < a.dim ? kp[row * kvs + kvh * a.dim + d] : krp[row * a.rot + d - a.dim]) << (16 * (j & 1));
                }
            }
        }
#pragma unroll
        for (int i = 0; i < NV; ++i) {  // (S and every sequence's key base are multiples of 8: 16-byte loads)
            const int at = tid + NT * i, v = at / CV, c0 = (at % CV) * 8;
            vreg[i] = *reinterpret_cast<const u32x4*>(vp + (size_t)min(v, a.vdim - 1) * a.S + min(sq.k0 + kt + c0, a.S - 8));
        }
    };
    static_assert((BN * CK) % NT == 0 && (DVP * CV) % NT == 0, "whole staging rounds");
    const int wq0 = sq.start + q_first + wave * NQ * 16;  // the wave's first query position
    const bool whole = q_first + (wave + 1) * NQ * 16 <= sq.nq;
    int kt = (first - sq.klo) / BN * BN;
    fetch(kt);
    for (; sq.klo + kt <= last; kt += BN) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NK; ++i) {
            const int at = tid + NT * i, d0 = (at % CK) * 8;
            *reinterpret_cast<u32x4*>(ks + (at / CK) * LK + d0) = !VEC || d0 < dq ? kreg[i] : u32x4{0u, 0u, 0u, 0u};
        }
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            const int at = tid + NT * i, c0 = (at % CV) * 8;
            *reinterpret_cast<u32x4*>(vs + (at / CV) * LV + c0) = at / CV < a.vdim && sq.k0 + kt + c0 < a.S ? vreg[i] : u32x4{0u, 0u, 0u, 0u};
        }
        __syncthreads();
        if (sq.klo + kt + BN <= last) fetch(kt + BN);
        f32x4 s[NQ][KT];
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
            for (int n = 0; n < NQ; ++n) s[n][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < KT; ++t)
#pragma unroll
            for (int q = 0; q < KS; ++q) {
                const u32x4 kf = *reinterpret_cast<const u32x4*>(ks + (t * 16 + l16) * LK + q * 32 + g * 8);
#pragma unroll
                for (int n = 0; n < NQ; ++n) s[n][t] = mfma16<BF16>(kf, qf[n][q], s[n][t]);
            }
        const int k_first = sq.klo + kt;
        // every query of the wave sees every key of the tile: no masks
        const bool open = whole && k_first + BN - 1 <= wq0 && k_first > wq0 + NQ * 16 - 1 - a.window;
        float ms[NQ], top[NQ];
        bool grown = false;
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
#pragma unroll
            for (int t = 0; t < KT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    s[n][t][r] *= sc;
                    if constexpr (CAP != kCapNone) s[n][t][r] = soft_cap2(s[n][t][r], cl2);
                }
            if (!open) {
#pragma unroll
                for (int t = 0; t < KT; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int kpos = k_first + t * 16 + g * 4 + r;
                        s[n][t][r] = kpos <= qpos[n] && kpos > qpos[n] - a.window ? s[n][t][r] : -INFINITY;
                    }
            }
            float mx = -INFINITY;
            if constexpr (CAP != kCapBounded) {
#pragma unroll
                for (int t = 0; t < KT; ++t)
#pragma unroll
                    for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[n][t][r]);
            }
            if constexpr (CAP != kCapBounded) {
                mx = fmaxf(mx, __shfl_xor(mx, 16));
                top[n] = fmaxf(mx, __shfl_xor(mx, 32));
                grown = grown || top[n] > m[n] + kStaleMax;
            }
        }
        if (CAP != kCapBounded && __any(grown)) {
#pragma unroll
            for (int n = 0; n < NQ; ++n) {
                const float now = fmaxf(m[n], top[n]), al = now == -INFINITY ? 1.0f : exp2_fast(m[n] - now);
                m[n] = now;
                l[n] *= al;
#pragma unroll
                for (int v = 0; v < VT; ++v) o[n][v] *= al;
            }
        }
#pragma unroll
        for (int n = 0; n < NQ; ++n) ms[n] = CAP == kCapBounded || m[n] == -INFINITY ? 0.0f : m[n];
#pragma unroll
        for (int b = 0; b < BN / 32; ++b) {
            u32x4 ph[NQ], pl[NQ];
#pragma unroll
            for (int n = 0; n < NQ; ++n)
#pragma unroll
                for (int j = 0; j < 4; ++j) {  // word j of the operand: keys 2j, 2j + 1 of the lane's eight (tile 2b, then tile 2b + 1)
                    const float p0 = exp2_fast(s[n][2 * b + (j >> 1)][2 * (j & 1)] - ms[n]), p1 = exp2_fast(s[n][2 * b + (j >> 1)][2 * (j & 1) + 1] - ms[n]);
                    uint32_t hi, lo;
                    split16x2<BF16>(p0, p1, hi, lo);
                    ph[n][j] = hi;
                    pl[n][j] = lo;
                    l[n] += p0 + p1;
                }
#pragma unroll
            for (int v = 0; v < VT; ++v) {
                const uint16_t* base = vs + (v * 16 + l16) * LV + b * 32 + g * 4;
                const u32x2 w0 = *reinterpret_cast<const u32x2*>(base), w1 = *reinterpret_cast<const u32x2*>(base + 16);
                const u32x4 vf = {w0[0], w0[1], w1[0], w1[1]};
#pragma unroll
                for (int n = 0; n < NQ; ++n) {
                    o[n][v] = mfma16<BF16>(vf, ph[n], o[n][v]);
                    o[n][v] = mfma16<BF16>(vf, pl[n], o[n][v]);
                }
            }
        }
    }
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        float lt = l[n] + __shfl_xor(l[n], 16);
        lt += __shfl_xor(lt, 32);
        if (a.sink) lt += exp2f(sink2 - m[n]);
        if (qpos[n] < 0) continue;
        const float inv = 1.0f / lt;
        const size_t t = (size_t)(sq.q0 + qpos[n] - sq.start);
        uint16_t* out = reinterpret_cast<uint16_t*>(a.out) + t * a.ldo + head * a.vdim;
        const uint16_t* gt = a.gate ? reinterpret_cast<const uint16_t*>(a.gate) + t * a.ldg + head * a.vdim : nullptr;
        const bool ovec = !(a.vdim & 3) && !(a.ldo & 3) && !(a.ldg & 3);
#pragma unroll
        for (int v = 0; v < VT; ++v) {
            const int d = v * 16 + g * 4;
            if (d >= a.vdim) continue;
            if (ovec) {
                float r[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) r[j] = o[n][v][j] * inv;
                if (gt) {
                    const u32x2 gw = *reinterpret_cast<const u32x2*>(gt + d);
#pragma unroll
                    for (int j = 0; j < 4; ++j) r[j] *= sigmoid_f(bits_to_float(j & 1 ? gw[j >> 1] >> 16 : gw[j >> 1] & 0xFFFFu, BF16));
                }
                *reinterpret_cast<u32x2*>(out + d) = u32x2{(uint32_t)float_to_bits<BF16>(r[0]) | ((uint32_t)float_to_bits<BF16>(r[1]) << 16),
                                                           (uint32_t)float_to_bits<BF16>(r[2]) | ((uint32_t)float_to_bits<BF16>(r[3]) << 16)};
            } else {
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (d + j < a.vdim) out[d + j] = float_to_bits<BF16>(o[n][v][j] * inv * (gt ? sigmoid_f(bits_to_float(gt[d + j], BF16)) : 1.0f));
            }
        }
    }
}

// Queries per workgroup: NT / 4.  Head sizes: q . k up to 256; values up to 256, a workgroup of 512 threads 128.  Bound by the one workgroup a CU holds
// (160 registers, eight waves): products, softmax and LDS reads of a tile hardly overlap.  3000 tokens of 3 to 5 requests, 32 heads: q . k 192
// and values 128 134 -> 103 us, 128 and 128 with bounded scores 155 -> 89, of which the order of the tiles 25.  Tried and slower: 32 queries a
// wave (twice the operands' use, 256 registers: 116 and 90), 64 queries a workgroup (142, 88), two workgroups a CU (spills: 138).
template <bool BF16, int NT, int CAP>
int launch_prompt(const PromptAttentionArgs& a, const int n_tiles, hipStream_t st) {
    const int dq = a.dim + a.rot;
    if ((long long)a.heads * n_tiles > 0x7FFFFFFFll) return TEAL_ERR_SHAPE;
    const dim3 grid(a.heads * n_tiles), block(NT);
#define TEAL_LP(DQ, DV, BN, VEC) do { hipLaunchKernelGGL((prompt_attention_kernel<BF16, DQ, DV, 1, BN, NT, CAP, VEC>), grid, block, 0, st, a); return launched(); } while (0)
    // (capped scores come with values no wider than the keys: fewer combinations)
#define TEAL_LP_V(DQ)                                                                                                   \
    do {                                                                                                               \
        if constexpr (CAP == kCapNone || DQ == 64) { if (a.vdim <= 64) TEAL_LP(DQ, 64, 64, true); }                    \
        if constexpr (CAP == kCapNone || DQ >= 128) { if (a.vdim <= 128) TEAL_LP(DQ, 128, 64, true); }                 \
        if constexpr (NT == 256 && (CAP == kCapNone || DQ > 128)) TEAL_LP(DQ, 256, 32, true);                            \
        return TEAL_ERR_SHAPE;                                                                                         \
    } while (0)
    if (dq > 256) return TEAL_ERR_SHAPE;
    if ((a.dim | a.rot | a.ldq) & 7) {  // any sizes, element by element
        if (a.vdim <= 128) { if (dq <= 128) TEAL_LP(128, 128, 64, false); TEAL_LP(256, 128, 64, false); }
        if constexpr (NT == 256) TEAL_LP(256, 256, 32, false);
        return TEAL_ERR_SHAPE;
    }
    if (dq <= 64) TEAL_LP_V(64);
    else if (dq <= 128) TEAL_LP_V(128);
    else if (dq <= 192) TEAL_LP_V(192);
    TEAL_LP_V(256);
#undef TEAL_LP_V
#undef TEAL_LP
}

// soft-capped scores (a.softcap > 0, vdim <= dim + rot); tile = 64 or 128 queries
int launch_prompt_capped(const PromptAttentionArgs& a, int tile, int n_tiles, int dtype, hipStream_t st);

}  // namespace teal
