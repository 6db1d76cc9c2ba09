// teal_prompt.hip — what stands between the matrix products of a Llama prompt pass of any length (teal_amd/gpt_fast/prefill.py:
// PromptPass), 16-bit rows [token][feature].  gfx950 / CDNA4, wave64.
//
//   prompt_norm_kernel       h = embedding row | h + y, x = RMSNorm(h) * w   (gpt-fast/model.py:158-161, 289-291)
//   prompt_rope_kernel       rotation of q in place, of k into its cache row; v into its cache row   (model.py:170-178)
//   prompt_attention16_kernel  softmax(q K^T / sqrt(d)) V of every token over the cached rows up to its position   (model.py:179-186)
//   silu_mul_kernel          silu(gate) * up   (model.py:258-259)
// Op by op these were some twenty launches per layer, every one a pass over the activations, and a library attention that read an
// explicit mask of tokens x cache rows: Llama-3-8B widths, 3000 tokens, per layer 560 us of row kernels and 1116 us of attention, now 103 (18 + 14
// + 18 + 43 us + the cache writes, 3.5 - 4 TB/s) and 122 us (74 useful GFLOP: 0.61 PFLOP/s); Llama-2-7B, 301 tokens, 55 launches -> 10.
#include "teal_prompt_attention.h"

namespace teal {

template <bool BF16>
__device__ __forceinline__ void unpack8(const u32x4 w, float (&o)[8]) {
#pragma unroll
    for (int j = 0; j < 4; ++j) { o[2 * j] = bits_to_float(w[j] & 0xFFFFu, BF16); o[2 * j + 1] = bits_to_float(w[j] >> 16, BF16); }
}
template <bool BF16>
__device__ __forceinline__ u32x4 pack8(const float (&v)[8]) {
    u32x4 w;
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = (uint32_t)float_to_bits<BF16>(v[2 * j]) | ((uint32_t)float_to_bits<BF16>(v[2 * j + 1]) << 16);
    return w;
}

struct PromptNormArgs {
    const uint16_t* emb;   // or null: [vocab][D]
    const void* tokens;    // with emb: int32 or int64 [T]
    uint16_t* h;           // [T][D] residual, updated in place
    const uint16_t* y;     // or null: 16-bit [T][D]
    const float* slabs;    // or null: fp32 [nslabs][T][D], added in slab order and rounded
    const uint16_t* w;     // [D]
    uint16_t* x;           // [T][D]
    unsigned* zero;        // or null: nzero counters to clear
    int D, vocab, tok64, nslabs, nzero;
    float eps;
};

// one workgroup per token, a thread holds up to two 16-byte pieces of the row.  The rounding points are the module path's 16-bit tensors
template <bool BF16, int NT>
__global__ __launch_bounds__(NT) void prompt_norm_kernel(const PromptNormArgs a) {
    constexpr int R = 2;
    __shared__ float red[NT / 64];
    const int tid = threadIdx.x, T = gridDim.x;
    const size_t t = blockIdx.x;
    if (t == 0 && tid < a.nzero) a.zero[tid] = 0u;
    float v[R][8], ss = 0.0f;
#pragma unroll
    for (int i = 0; i < R; ++i) {
        const int d = (tid + NT * i) * 8;
        if (d >= a.D) continue;
        if (a.emb) {
            const long long id = a.tok64 ? reinterpret_cast<const long long*>(a.tokens)[t] : (long long)reinterpret_cast<const int*>(a.tokens)[t];
            const size_t row = (size_t)(id < 0 ? 0 : id >= a.vocab ? a.vocab - 1 : id);
            unpack8<BF16>(*reinterpret_cast<const u32x4*>(a.emb + row * a.D + d), v[i]);
        } else {
            unpack8<BF16>(*reinterpret_cast<const u32x4*>(a.h + t * a.D + d), v[i]);
        }
        if (a.slabs || a.y) {
            float y[8];
            if (a.slabs) {
#pragma unroll
                for (int j = 0; j < 8; ++j) y[j] = 0.0f;
                for (int k = 0; k < a.nslabs; ++k) {
                    const float* p = a.slabs + ((size_t)k * T + t) * a.D + d;
                    const f32x4 s0 = *reinterpret_cast<const f32x4*>(p), s1 = *reinterpret_cast<const f32x4*>(p + 4);
#pragma unroll
                    for (int j = 0; j < 4; ++j) { y[j] += s0[j]; y[4 + j] += s1[j]; }
                }
#pragma unroll
                for (int j = 0; j < 8; ++j) y[j] = bits_to_float(float_to_bits<BF16>(y[j]), BF16);
            } else {
                unpack8<BF16>(*reinterpret_cast<const u32x4*>(a.y + t * a.D + d), y);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) v[i][j] = bits_to_float(float_to_bits<BF16>(v[i][j] + y[j]), BF16);
        }
        if (a.emb || a.slabs || a.y) *reinterpret_cast<u32x4*>(a.h + t * a.D + d) = pack8<BF16>(v[i]);
#pragma unroll
        for (int j = 0; j < 8; ++j) ss = fmaf(v[i][j], v[i][j], ss);
    }
    const float rstd = rsqrtf(block_sum<NT>(ss, red, tid) / (float)a.D + a.eps);
#pragma unroll
    for (int i = 0; i < R; ++i) {
        const int d = (tid + NT * i) * 8;
        if (d >= a.D) continue;
        float w[8];
        unpack8<BF16>(*reinterpret_cast<const u32x4*>(a.w + d), w);
#pragma unroll
        for (int j = 0; j < 8; ++j) w[j] *= bits_to_float(float_to_bits<BF16>(v[i][j] * rstd), BF16);
        *reinterpret_cast<u32x4*>(a.x + t * a.D + d) = pack8<BF16>(w);
    }
}

// a position of the prompt, kept inside the cache
__device__ __forceinline__ int prompt_pos(const void* pos, const int pos64, const int t, const int max_seq) {
    const long long p = pos64 ? reinterpret_cast<const long long*>(pos)[t] : (long long)reinterpret_cast<const int*>(pos)[t];
    return (int)(p < 0 ? 0 : p >= max_seq ? max_seq - 1 : p);
}

struct PromptRopeArgs {
    uint16_t* qkv;        // [T][ldq]: q | k | v
    const uint16_t* rope; // (cos, sin) [positions][hd / 2][2]
    const void* pos;      // int32 or int64 [T]
    uint16_t* kc;         // [n_kv][max_seq][hd]
    uint16_t* vc;
    int ldq, pos64, n_head, n_kv, hd, max_seq;
};

// eight elements of a token's row per thread
template <bool BF16>
__global__ __launch_bounds__(256) void prompt_rope_kernel(const PromptRopeArgs a) {
    const int t = blockIdx.x, c = (blockIdx.y * 256 + threadIdx.x) * 8, nq = a.n_head * a.hd, nkv = a.n_kv * a.hd;
    if (c >= nq + 2 * nkv) return;
    const int p = prompt_pos(a.pos, a.pos64, t, a.max_seq);
    uint16_t* src = a.qkv + (size_t)t * a.ldq + c;
    const u32x4 raw = *reinterpret_cast<const u32x4*>(src);
    if (c >= nq + nkv) {
        const int h = (c - nq - nkv) / a.hd, d = (c - nq - nkv) % a.hd;
        *reinterpret_cast<u32x4*>(a.vc + ((size_t)h * a.max_seq + p) * a.hd + d) = raw;
        return;
    }
    const bool isk = c >= nq;
    const int h = (isk ? c - nq : c) / a.hd, d = (isk ? c - nq : c) % a.hd;
    float x[8], cs[8];
    unpack8<BF16>(raw, x);
    unpack8<BF16>(*reinterpret_cast<const u32x4*>(a.rope + (size_t)p * a.hd + d), cs);
#pragma unroll
    for (int j = 0; j < 8; j += 2) {
        const float e = rope_even(x[j], x[j + 1], cs[j], cs[j + 1]), o = rope_odd(x[j], x[j + 1], cs[j], cs[j + 1]);
        x[j] = e;
        x[j + 1] = o;
    }
    *reinterpret_cast<u32x4*>(isk ? a.kc + ((size_t)h * a.max_seq + p) * a.hd + d : src) = pack8<BF16>(x);
}

struct PromptAttention16Args {
    const uint16_t* q;    // [T][ldq], rotated
    const uint16_t* kc;   // [n_kv][max_seq][hd]
    const uint16_t* vc;
    const void* pos;
    uint16_t* out;        // [T][ldo]
    int ldq, ldo, T, pos64, rep, max_seq;
    float scale2;         // scale in log2 units
};

// Flash attention of 128 queries per workgroup over 64-row tiles of the cache as it is.  S^T = K Q^T and O^T = V^T P^T: a lane holds four
// consecutive keys of one query after the first product, which is its operand of the second; V comes transposed out of the LDS
// (ds_read_b64_tr_b16), so neither the weights nor V cross lanes or memory.  A wave takes 32 queries: at 16 every operand read from the
// LDS would serve one product, and the LDS, not the matrix cores, would be the limit (128 bytes per clock against 256 wanted).  The
// running maximum is replaced only when a score exceeds it by kStaleMax (weights up to 2^8 then, which changes nothing in their relative
// precision): rescaling the accumulators costs as much as a quarter of the products.
template <bool BF16, int HD>
__global__ __launch_bounds__(256, 2) void prompt_attention16_kernel(const PromptAttention16Args a) {
    constexpr int NQ = 2, BM = 128, BN = 64, KS = HD / 32, KT = BN / 16, VT = HD / 16, LK = HD + 8, LV = HD + 16, NT = 256, CH = HD / 8, NL = BN * CH / NT;
    __shared__ __align__(16) uint16_t ks[BN * LK];
    __shared__ __align__(16) uint16_t vs[BN * LV];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l16 = lane & 15, g = lane >> 4;
    const int head = blockIdx.x, q0 = (gridDim.y - 1 - blockIdx.y) * BM + wave * 32;  // (the late tiles are the long ones: first)
    const uint16_t* kp = a.kc + (size_t)(head / a.rep) * a.max_seq * HD;
    const uint16_t* vp = a.vc + (size_t)(head / a.rep) * a.max_seq * HD;
    u32x4 qf[NQ][KS];
    int qpos[NQ], lo = 0x7FFFFFFF, hi = -1;
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        const int qi = q0 + 16 * n + l16, at = min(qi, a.T - 1);
        qpos[n] = qi < a.T ? prompt_pos(a.pos, a.pos64, at, a.max_seq) : -1;
        lo = min(lo, qpos[n]);
        hi = max(hi, qpos[n]);
#pragma unroll
        for (int s = 0; s < KS; ++s) qf[n][s] = *reinterpret_cast<const u32x4*>(a.q + (size_t)at * a.ldq + head * HD + s * 32 + g * 8);
    }
#pragma unroll
    for (int d = 1; d < 16; d <<= 1) { lo = min(lo, __shfl_xor(lo, d)); hi = max(hi, __shfl_xor(hi, d)); }  // the wave's first and last position
    lo = __builtin_amdgcn_readfirstlane(lo);
    hi = __builtin_amdgcn_readfirstlane(hi);
    __shared__ int last_of[4];
    if (lane == 0) last_of[wave] = hi;
    __syncthreads();
    const int last = max(max(last_of[0], last_of[1]), max(last_of[2], last_of[3]));
    float m[NQ], l[NQ];
    f32x4 o[NQ][VT];
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        m[n] = -INFINITY;
        l[n] = 0.0f;
#pragma unroll
        for (int v = 0; v < VT; ++v) o[n][v] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    u32x4 kreg[NL], vreg[NL];
    auto fetch = [&](const int kt) {  // (rows past the cache's end repeat its last one: they are masked)
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int at = tid + NT * i;
            const size_t off = (size_t)min(kt + at / CH, a.max_seq - 1) * HD + (at % CH) * 8;
            kreg[i] = *reinterpret_cast<const u32x4*>(kp + off);
            vreg[i] = *reinterpret_cast<const u32x4*>(vp + off);
        }
    };
    fetch(0);
    for (int kt = 0; kt <= last; kt += BN) {
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NL; ++i) {
            const int at = tid + NT * i;
            *reinterpret_cast<u32x4*>(ks + (at / CH) * LK + (at % CH) * 8) = kreg[i];
            *reinterpret_cast<u32x4*>(vs + (at / CH) * LV + (at % CH) * 8) = vreg[i];
        }
        __syncthreads();
        if (kt + BN <= last) fetch(kt + BN);
        if (kt > hi) continue;  // (wave-uniform: nothing here for this wave's queries)
        f32x4 s[NQ][KT];
#pragma unroll
        for (int t = 0; t < KT; ++t) {
#pragma unroll
            for (int n = 0; n < NQ; ++n) s[n][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < KS; ++q) {
                const u32x4 kf = *reinterpret_cast<const u32x4*>(ks + (t * 16 + l16) * LK + q * 32 + g * 8);
#pragma unroll
                for (int n = 0; n < NQ; ++n) s[n][t] = mfma16<BF16>(kf, qf[n][q], s[n][t]);
            }
        }
        const bool open = kt + BN - 1 <= lo;  // every query of the wave sees every key of the tile
        bool grown = false;
        float mx[NQ];
#pragma unroll
        for (int n = 0; n < NQ; ++n) {
            float top = -INFINITY;
#pragma unroll
            for (int t = 0; t < KT; ++t)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    float v = s[n][t][r] * a.scale2;
                    if (!open) v = kt + t * 16 + g * 4 + r <= qpos[n] ? v : -INFINITY;
                    s[n][t][r] = v;
                    top = fmaxf(top, v);
                }
            top = fmaxf(top, __shfl_xor(top, 16));
            top = fmaxf(top, __shfl_xor(top, 32));
            mx[n] = top;
            grown = grown || top > m[n] + kStaleMax;
        }
        if (__any(grown)) {
#pragma unroll
            for (int n = 0; n < NQ; ++n) {
                const float now = fmaxf(m[n], mx[n]), al = now == -INFINITY ? 1.0f : exp2_fast(m[n] - now);
                m[n] = now;
                l[n] *= al;
#pragma unroll
                for (int v = 0; v < VT; ++v) o[n][v] *= al;
            }
        }
        float ms[NQ];
#pragma unroll
        for (int n = 0; n < NQ; ++n) ms[n] = m[n] == -INFINITY ? 0.0f : m[n];
#pragma unroll
        for (int b = 0; b < BN / 32; ++b) {
            u32x4 ph[NQ];
#pragma unroll
            for (int n = 0; n < NQ; ++n)
#pragma unroll
                for (int j = 0; j < 4; ++j) {  // word j: keys 2j, 2j + 1 of the lane's eight (tile 2b, then tile 2b + 1)
                    const float p0 = exp2_fast(s[n][2 * b + (j >> 1)][2 * (j & 1)] - ms[n]), p1 = exp2_fast(s[n][2 * b + (j >> 1)][2 * (j & 1) + 1] - ms[n]);
                    ph[n][j] = (uint32_t)float_to_bits<BF16>(p0) | ((uint32_t)float_to_bits<BF16>(p1) << 16);
                    l[n] += p0 + p1;
                }
#pragma unroll
            for (int v = 0; v < VT; ++v) {
                const uint16_t* base = vs + (b * 32 + g * 4 + (l16 >> 2)) * LV + v * 16 + 4 * (l16 & 3);
                const u32x2 w0 = lds_column4(base), w1 = lds_column4(base + 16 * LV);
                const u32x4 vf = {w0[0], w0[1], w1[0], w1[1]};
#pragma unroll
                for (int n = 0; n < NQ; ++n) o[n][v] = mfma16<BF16>(vf, ph[n], o[n][v]);
            }
        }
    }
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
        float lt = l[n] + __shfl_xor(l[n], 16);
        lt += __shfl_xor(lt, 32);
        if (qpos[n] < 0) continue;
        const float inv = 1.0f / lt;
        uint16_t* out = a.out + (size_t)(q0 + 16 * n + l16) * a.ldo + head * HD + g * 4;
#pragma unroll
        for (int v = 0; v < VT; ++v)
            *reinterpret_cast<u32x2*>(out + v * 16) = u32x2{(uint32_t)float_to_bits<BF16>(o[n][v][0] * inv) | ((uint32_t)float_to_bits<BF16>(o[n][v][1] * inv) << 16),
                                                            (uint32_t)float_to_bits<BF16>(o[n][v][2] * inv) | ((uint32_t)float_to_bits<BF16>(o[n][v][3] * inv) << 16)};
    }
}

// h = round(silu(gate)) * up (the module path's rounding points), eight elements per thread
template <bool BF16>
__global__ __launch_bounds__(256) void silu_mul_kernel(const uint16_t* __restrict__ gate, const uint16_t* __restrict__ up, uint16_t* __restrict__ h, const size_t n8) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n8) return;
    float x[8], u[8];
    unpack8<BF16>(__builtin_nontemporal_load(reinterpret_cast<const u32x4*>(gate) + i), x);
    unpack8<BF16>(__builtin_nontemporal_load(reinterpret_cast<const u32x4*>(up) + i), u);
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = bits_to_float(float_to_bits<BF16>(x[j] * sigmoid_f(x[j])), BF16) * u[j];
    reinterpret_cast<u32x4*>(h)[i] = pack8<BF16>(x);
}

}  // namespace teal

using namespace teal;

extern "C" {

int teal_prompt_norm(const void* emb, int vocab, const void* tokens, int tokens64, void* h, const void* y, const float* slabs, int n_slabs, const void* w, void* x, int T, int dim,
                     float eps, unsigned* zero, int n_zero, int dtype, void* stream) {
    if (!h || !w || !x || T <= 0 || dim <= 0 || (!emb) != (!tokens) || (emb && vocab <= 0) || (y && slabs) || (slabs && n_slabs < 1) || (zero && (n_zero < 1 || n_zero > 256)))
        return TEAL_ERR_ARG;
    if (dtype != TEAL_F16 && dtype != TEAL_BF16) return TEAL_ERR_DTYPE;
    if ((dim & 7) || dim > 16384) return TEAL_ERR_SHAPE;
    const void* ps[] = {emb, h, y, slabs, w, x};
    for (const void* p : ps)
        if (!aligned16(p)) return TEAL_ERR_ALIGN;
    const PromptNormArgs a = {reinterpret_cast<const uint16_t*>(emb), tokens, reinterpret_cast<uint16_t*>(h), reinterpret_cast<const uint16_t*>(y), slabs,
                              reinterpret_cast<const uint16_t*>(w), reinterpret_cast<uint16_t*>(x), zero, dim, vocab, tokens64, slabs ? n_slabs : 0, zero ? n_zero : 0, eps};
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
#define TEAL_PN(BF, NT) hipLaunchKernelGGL((prompt_norm_kernel<BF, NT>), dim3(T), dim3(NT), 0, st, a)
#define TEAL_PN_D(BF) do { if (dim <= 4096) TEAL_PN(BF, 256); else if (dim <= 8192) TEAL_PN(BF, 512); else TEAL_PN(BF, 1024); } while (0)
    if (dtype == TEAL_BF16) TEAL_PN_D(true); else TEAL_PN_D(false);
#undef TEAL_PN_D
#undef TEAL_PN
    return launched();
}

int teal_prompt_rope(void* qkv, int ldq, const void* rope, const void* pos, int pos64, void* k_cache, void* v_cache, int T, int n_head, int n_kv_head, int head_dim, int max_seq,
                     int dtype, void* stream) {
    if (!qkv || !rope || !pos || !k_cache || !v_cache || T <= 0) return TEAL_ERR_ARG;
    if (dtype != TEAL_F16 && dtype != TEAL_BF16) return TEAL_ERR_DTYPE;
    if (n_head <= 0 || n_kv_head <= 0 || head_dim <= 0 || (head_dim & 7) || max_seq <= 0 || (ldq & 7) || ldq < (n_head + 2 * n_kv_head) * head_dim) return TEAL_ERR_SHAPE;
    const void* ps[] = {qkv, rope, k_cache, v_cache};
    for (const void* p : ps)
        if (!aligned16(p)) return TEAL_ERR_ALIGN;
    const PromptRopeArgs a = {reinterpret_cast<uint16_t*>(qkv), reinterpret_cast<const uint16_t*>(rope), pos, reinterpret_cast<uint16_t*>(k_cache),
                              reinterpret_cast<uint16_t*>(v_cache), ldq, pos64, n_head, n_kv_head, head_dim, max_seq};
    const dim3 grid(T, ((n_head + 2 * n_kv_head) * head_dim / 8 + 255) / 256);
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (dtype == TEAL_BF16) hipLaunchKernelGGL((prompt_rope_kernel<true>), grid, dim3(256), 0, st, a);
    else hipLaunchKernelGGL((prompt_rope_kernel<false>), grid, dim3(256), 0, st, a);
    return launched();
}

int teal_prompt_attention(const void* q, int ldq, const void* k_cache, const void* v_cache, const void* pos, int pos64, void* out, int ldo, int T, int n_head, int n_kv_head,
                          int head_dim, int max_seq, float scale, int dtype, void* stream) {
    if (!q || !k_cache || !v_cache || !pos || !out || T <= 0) return TEAL_ERR_ARG;
    if (dtype != TEAL_F16 && dtype != TEAL_BF16) return TEAL_ERR_DTYPE;
    if ((head_dim != 64 && head_dim != 128) || n_head <= 0 || n_kv_head <= 0 || n_head % n_kv_head || max_seq <= 0 || (ldq & 7) || ldq < n_head * head_dim || (ldo & 3) ||
        ldo < n_head * head_dim || T > 65535 * 128)
        return TEAL_ERR_SHAPE;
    const void* ps[] = {q, k_cache, v_cache, out};
    for (const void* p : ps)
        if (!aligned16(p)) return TEAL_ERR_ALIGN;
    const PromptAttention16Args a = {reinterpret_cast<const uint16_t*>(q), reinterpret_cast<const uint16_t*>(k_cache), reinterpret_cast<const uint16_t*>(v_cache), pos,
                                     reinterpret_cast<uint16_t*>(out), ldq, ldo, T, pos64, n_head / n_kv_head, max_seq, scale * kLog2e};
    const dim3 grid(n_head, (T + 127) / 128);
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
#define TEAL_PA(BF, HDV) hipLaunchKernelGGL((prompt_attention16_kernel<BF, HDV>), grid, dim3(256), 0, st, a)
    if (dtype == TEAL_BF16) { if (head_dim == 128) TEAL_PA(true, 128); else TEAL_PA(true, 64); }
    else { if (head_dim == 128) TEAL_PA(false, 128); else TEAL_PA(false, 64); }
#undef TEAL_PA
    return launched();
}

int teal_silu_mul(const void* gate, const void* up, void* h, size_t n, int dtype, void* stream) {
    if (!gate || !up || !h || n == 0) return TEAL_ERR_ARG;
    if (dtype != TEAL_F16 && dtype != TEAL_BF16) return TEAL_ERR_DTYPE;
    if (n & 7) return TEAL_ERR_SHAPE;
    if (!aligned16(gate) || !aligned16(up) || !aligned16(h)) return TEAL_ERR_ALIGN;
    const size_t n8 = n / 8;
    const dim3 grid((unsigned)((n8 + 255) / 256));
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    auto* gp = reinterpret_cast<const uint16_t*>(gate);
    auto* up_ = reinterpret_cast<const uint16_t*>(up);
    if (dtype == TEAL_BF16) hipLaunchKernelGGL((silu_mul_kernel<true>), grid, dim3(256), 0, st, gp, up_, reinterpret_cast<uint16_t*>(h), n8);
    else hipLaunchKernelGGL((silu_mul_kernel<false>), grid, dim3(256), 0, st, gp, up_, reinterpret_cast<uint16_t*>(h), n8);
    return launched();
}

}  // extern "C"
