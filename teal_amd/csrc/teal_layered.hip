// teal_layered.hip — row kernels of the layered decoder designs (teal_amd/gpt_fast/layered.py): what stands between two matrix
// products of a block, with the residual stream held in fp32.  gfx950 / CDNA4, wave64; fp16, bf16 and true 32-bit activations.
//
//   resid_norm_kernel   x = embedding row | x + [post norm](y + bias), then h = RMSNorm(x) * w   (one workgroup per token)
//   gated_act_kernel    h = act(gate + bias) * (up + bias)
//   softcap_kernel      logits -> fp32, cap * tanh(logits / cap)
//   sample_rows_kernel  one token per row of fp32 logits: top-k filter, softmax, exponential race (or the largest logit)
#include "teal_layered.h"

namespace teal {

struct ResidNormArgs {
    float* x;               // residual stream [rows][D], updated in place
    const int32_t* tokens;  // or null: x = embed[tokens[row]]
    const void* embed;      // [vocab][D]
    const void* y;          // or null: sublayer output [rows][ldy]
    const void* y_bias;     // or null: [D], added to y
    const void* post_w;     // or null: y is RMS-normed with this weight before it joins the residual
    const void* pre_w;      // or null: h = RMSNorm(x) * pre_w
    void* h;                // [launch rows][D]
    const int32_t* rows;    // or null: row of x / y / tokens a workgroup handles (a subset of the rows); h is packed
    int D, ldy, vocab;
    float eps, off;         // off: added to the norms' weights (weights stored around zero: 1)
    int nslabs, slab_rows;  // nslabs > 0: y is the sum of fp32 slabs [nslabs][slab_rows][ldy]
    unsigned* zero;         // or null: nzero counters to clear
    int nzero;
};

template <int DT, int NT, int VEC>
__global__ __launch_bounds__(NT) void resid_norm_kernel(const ResidNormArgs a) {
    using N = Num<DT>;
    using S = typename N::S;
    extern __shared__ __align__(16) unsigned char smem[];
    float* buf = reinterpret_cast<float*>(smem);  // [D]
    __shared__ float red[NT / 64];
    const int tid = threadIdx.x, D = a.D;
    const size_t row = a.rows ? (size_t)a.rows[blockIdx.x] : (size_t)blockIdx.x;
    if (blockIdx.x == 0 && tid < a.nzero) a.zero[tid] = 0u;
    float* x = a.x + row * D;
    const float* ys = reinterpret_cast<const float*>(a.y) + row * a.ldy;
    const S* y = a.y ? reinterpret_cast<const S*>(a.y) + row * a.ldy : nullptr;
    const S* yb = reinterpret_cast<const S*>(a.y_bias);
    const S* pw = reinterpret_cast<const S*>(a.post_w);
    const S* nw = reinterpret_cast<const S*>(a.pre_w);
    auto ldv = [](const S* p, float (&o)[VEC]) {
        if constexpr (VEC == 4 && DT != TEAL_F32) {
            const u32x2 w = *reinterpret_cast<const u32x2*>(p);
#pragma unroll
            for (int j = 0; j < 2; ++j) { o[2 * j] = bits_to_float(w[j] & 0xFFFFu, DT == TEAL_BF16); o[2 * j + 1] = bits_to_float(w[j] >> 16, DT == TEAL_BF16); }
        } else if constexpr (VEC == 4) {
            const f32x4 w = *reinterpret_cast<const f32x4*>(p);
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = w[j];
        } else {
            o[0] = N::ld(p);
        }
    };
    auto ldx = [](const float* p, float (&o)[VEC]) {
        if constexpr (VEC == 4) {
            const f32x4 w = *reinterpret_cast<const f32x4*>(p);
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = w[j];
        } else {
            o[0] = *p;
        }
    };
    auto stx = [](float* p, const float (&o)[VEC]) {
        if constexpr (VEC == 4) *reinterpret_cast<f32x4*>(p) = f32x4{o[0], o[1], o[2], o[3]};
        else *p = o[0];
    };
    float rstd_y = 1.0f;
    if (y) {
        float ss = 0.0f;
        for (int i = tid * VEC; i < D; i += NT * VEC) {
            float v[VEC];
            if (a.nslabs) {
                ldx(ys + i, v);
                for (int k = 1; k < a.nslabs; ++k) {
                    float u[VEC];
                    ldx(ys + (size_t)k * a.slab_rows * a.ldy + i, u);
#pragma unroll
                    for (int j = 0; j < VEC; ++j) v[j] += u[j];
                }
            } else {
                ldv(y + i, v);
            }
            if (yb) {
                float b[VEC];
                ldv(yb + i, b);
#pragma unroll
                for (int j = 0; j < VEC; ++j) v[j] += b[j];
            }
            stx(buf + i, v);  // (each thread reads back only what it wrote)
#pragma unroll
            for (int j = 0; j < VEC; ++j) ss = fmaf(v[j], v[j], ss);
        }
        if (pw) rstd_y = 1.0f / sqrtf(block_sum<NT>(ss, red, tid) / (float)D + a.eps);
    }
    const S* erow = nullptr;
    if (a.tokens) {
        const int t = min(max(a.tokens[row], 0), a.vocab - 1);
        erow = reinterpret_cast<const S*>(a.embed) + (size_t)t * D;
    }
    float ss = 0.0f;
    for (int i = tid * VEC; i < D; i += NT * VEC) {
        float v[VEC];
        if (erow) ldv(erow + i, v);
        else ldx(x + i, v);
        if (y) {
            float u[VEC];
            ldx(buf + i, u);
            if (pw) {
                float w[VEC];
                ldv(pw + i, w);
#pragma unroll
                for (int j = 0; j < VEC; ++j) u[j] = u[j] * rstd_y * (a.off + w[j]);
            }
#pragma unroll
            for (int j = 0; j < VEC; ++j) v[j] += u[j];
        }
        if (erow || y) stx(x + i, v);
        stx(buf + i, v);
#pragma unroll
        for (int j = 0; j < VEC; ++j) ss = fmaf(v[j], v[j], ss);
    }
    if (!nw) return;
    const float rstd = 1.0f / sqrtf(block_sum<NT>(ss, red, tid) / (float)D + a.eps);
    S* h = reinterpret_cast<S*>(a.h) + (size_t)blockIdx.x * D;
    for (int i = tid * VEC; i < D; i += NT * VEC) {
        float v[VEC], w[VEC];
        ldx(buf + i, v);
        ldv(nw + i, w);
        if constexpr (VEC == 4 && DT != TEAL_F32) {
            uint32_t o[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) o[j] = N::cvt(v[j] * rstd * (a.off + w[j]));
            *reinterpret_cast<u32x2*>(h + i) = u32x2{o[0] | (o[1] << 16), o[2] | (o[3] << 16)};
        } else {
#pragma unroll
            for (int j = 0; j < VEC; ++j) h[i + j] = N::cvt(v[j] * rstd * (a.off + w[j]));
        }
    }
}

// h[t][n] = act(gu[t][n] + bg[n]) [* (gu[t][up0 + n] + bu[n]), up0 > 0]; act 0 = silu, 1 = gelu (tanh form), 2 = squared relu
template <int DT>
__global__ __launch_bounds__(256) void gated_act_kernel(const typename Num<DT>::S* __restrict__ gu, const int ldg, const int up0,
                                                        const typename Num<DT>::S* __restrict__ bg, const typename Num<DT>::S* __restrict__ bu,
                                                        typename Num<DT>::S* __restrict__ h, const int ldh, const int F, const int act, const bool vec) {
    using N = Num<DT>;
    const size_t t = blockIdx.x;
    const int n0 = (blockIdx.y * 256 + threadIdx.x) * 8;
    if (n0 >= F) return;
    const typename N::S* g = gu + t * ldg;
    typename N::S* o = h + t * ldh;
    const int m = min(8, F - n0);
    float gv[8], uv[8], bgv[8], buv[8];
    if (m == 8) {
        ld8<DT>(g + n0, gv, vec);
        if (up0) ld8<DT>(g + up0 + n0, uv, vec);
        if (bg) ld8<DT>(bg + n0, bgv, vec);
        if (bu) ld8<DT>(bu + n0, buv, vec);
    } else {
        for (int j = 0; j < m; ++j) {
            gv[j] = N::ld(g + n0 + j);
            if (up0) uv[j] = N::ld(g + up0 + n0 + j);
            if (bg) bgv[j] = N::ld(bg + n0 + j);
            if (bu) buv[j] = N::ld(bu + n0 + j);
        }
    }
    typename N::S r[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float z = bg ? gv[j] + bgv[j] : gv[j];
        const float u = !up0 ? 1.0f : (bu ? uv[j] + buv[j] : uv[j]);
        r[j] = N::cvt((act == TEAL_ACT_RELU2 ? relu2_f(z) : (act == TEAL_ACT_GELU_TANH ? gelu_tanh_f(z) : z * sigmoid_f(z))) * u);
    }
    if (vec && m == 8 && DT != TEAL_F32) {
        u32x4 w;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = (uint32_t)r[2 * j] | ((uint32_t)r[2 * j + 1] << 16);
        *reinterpret_cast<u32x4*>(o + n0) = w;
    } else {
        for (int j = 0; j < m; ++j) o[n0 + j] = r[j];
    }
}

template <int DT>
__global__ __launch_bounds__(256) void softcap_kernel(const typename Num<DT>::S* __restrict__ in, const int ldi, float* __restrict__ out, const int V,
                                                      const float cap) {
    const int n = blockIdx.y * 256 + threadIdx.x;
    if (n >= V) return;
    const float v = Num<DT>::ld(in + (size_t)blockIdx.x * ldi + n);
    out[(size_t)blockIdx.x * V + n] = cap > 0.0f ? cap * tanhf(v / cap) : v;
}

// ------------------------------------------------------------------------------------------------
// Sampler over fp32 logits, one workgroup per row: the 16-bit samplers of teal_attention.hip for logits that are not rounded.  The
// k-th largest logit is found exactly: keys order like the floats, d = (largest key) - key; a 256-bin histogram of d >> sh covers the
// keys nearest to the maximum (the others do no atomics), widened until it holds k of them, then the pivot's bin is resolved eight
// bits at a time.  Ties at the pivot stay in.  The race is the one of the 16-bit samplers: argmax exp((x - max) / T) / Exp(1).
// ------------------------------------------------------------------------------------------------
__device__ __forceinline__ uint32_t order_key32(const float f) {
    const uint32_t b = __float_as_uint(f);
    return (b & 0x80000000u) ? ~b : (b | 0x80000000u);
}

// Bound by latency: five or so passes of one workgroup over its row.  PIECES > 0: the row is read once, 16 bytes at a time, and stays in registers
// (1024 x 4 PIECES logits; with 16 pieces the compiler does not keep them there: 65536 logits 167 us, from memory 60); 0: any size, stride and
// alignment, every pass reads memory.  32000 logits, top 200: 46 us from memory, 21 from registers; 8000: 19 and 12.
__device__ __forceinline__ float from_order_key32(const uint32_t k) { return __uint_as_float((k & 0x80000000u) ? (k & 0x7FFFFFFFu) : ~k); }

template <int PIECES>
__global__ __launch_bounds__(1024) void sample_rows_kernel(const float* __restrict__ logits, const int ld, const int V, const int top_k, const float inv_temp,
                                                           unsigned long long* __restrict__ rng, int32_t* __restrict__ token_out, int32_t* __restrict__ pos_inout,
                                                           int32_t* __restrict__ history, const int history_len) {
    __shared__ unsigned hist[256], sel[2];
    __shared__ float fred[16];
    __shared__ int ired[16];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, row = blockIdx.x;
    const float* x = logits + (size_t)row * ld;
    u32x4 own[PIECES > 0 ? PIECES : 1];  // logits, then their distances d from the largest: one register each, whatever a pass wants of them
    float mx = -INFINITY;
    if constexpr (PIECES > 0) {
#pragma unroll
        for (int p = 0; p < PIECES; ++p) own[p] = *reinterpret_cast<const u32x4*>(x + min(4 * (1024 * p + tid), V - 4));
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {  // (past the end: the last logits once more)
#pragma unroll
            for (int j = 0; j < 4; ++j) mx = fmaxf(mx, __uint_as_float(own[p][j]));
        }
    } else {
        for (int i = tid; i < V; i += 1024) mx = fmaxf(mx, x[i]);
    }
    mx = block_max<1024>(mx, fred, tid);
    const uint32_t kmax = order_key32(mx);
    if constexpr (PIECES > 0) {
#pragma unroll
        for (int p = 0; p < PIECES; ++p) {
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                own[p][j] = kmax - order_key32(__uint_as_float(own[p][j]));
                asm volatile("" : "+v"(own[p][j]));  // (or both forms are kept)
            }
        }
    }
    auto each = [&](auto f) {  // f(index, d) for the thread's logits
        if constexpr (PIECES > 0) {
#pragma unroll
            for (int p = 0; p < PIECES; ++p) {
                const int i = 4 * (1024 * p + tid);
                if (i < V) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) f(i + j, own[p][j]);
                }
            }
        } else {
            for (int i = tid; i < V; i += 1024) f(i, kmax - order_key32(x[i]));
        }
    };
    uint32_t limit = 0xFFFFFFFFu;  // keep keys with kmax - key <= limit
    if (top_k > 0 && top_k < V && inv_temp > 0.0f) {
        // histogram of (d - lo) >> sh for d in [lo, lo + (256 << sh)); leaves the bin of the need-th key in sel[0], its rank there in sel[1],
        // or sel[1] = 0 when the window holds fewer
        auto window = [&](const uint32_t lo, const int sh, const unsigned need) {
            if (tid < 256) hist[tid] = 0u;
            __syncthreads();
            each([&](int, const uint32_t d) {
                if (d >= lo && ((d - lo) >> sh) < 256u) atomicAdd(&hist[(d - lo) >> sh], 1u);
            });
            __syncthreads();
            if (tid < 64) {
                unsigned own = 0u;
#pragma unroll
                for (int j = 0; j < 4; ++j) own += hist[4 * tid + j];
                unsigned incl = own;
#pragma unroll
                for (int k = 1; k < 64; k <<= 1) {
                    const unsigned t = (unsigned)__shfl_up((int)incl, k);
                    if (tid >= k) incl += t;
                }
                unsigned before = incl - own;
                if (tid == 63 && incl < need) sel[1] = 0u;
                for (int j = 0; j < 4; ++j) {
                    const unsigned h = hist[4 * tid + j];
                    if (before < need && before + h >= need) { sel[0] = 4u * tid + j; sel[1] = need - before; }
                    before += h;
                }
            }
            __syncthreads();
        };
        int sh = 14;
        window(0u, sh, (unsigned)top_k);
        while (sel[1] == 0u && sh < 24) {  // (at sh = 24 the window is every key)
            sh = min(sh + 5, 24);
            __syncthreads();
            window(0u, sh, (unsigned)top_k);
        }
        uint32_t lo = sel[0] << sh;
        unsigned need = sel[1];
        while (sh > 0) {
            const int step = min(8, sh);
            __syncthreads();
            window(lo, sh - step, need);  // (bins past this one's end hold keys of the next: the need-th key comes before them)
            sh -= step;
            lo += sel[0] << sh;
            need = sel[1];
        }
        limit = lo;
    }
    const uint32_t seed = (uint32_t)rng[2 * row], ctr = (uint32_t)rng[2 * row + 1];
    float best = -INFINITY;
    int besti = 0x7FFFFFFF;
    each([&](const int i, const uint32_t d) {
        if (d > limit) return;
        const float v = from_order_key32(kmax - d);
        float sc = v;
        if (inv_temp > 0.0f) {
            const float u = ((float)(hash3(seed, ctr, (uint32_t)i) >> 8) + 0.5f) * (1.0f / 16777216.0f);
            sc = expf((v - mx) * inv_temp) / (-logf(u));
        }
        if (sc > best || (sc == best && i < besti)) { best = sc; besti = i; }
    });
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        const float ob = __shfl_xor(best, d);
        const int oi = __shfl_xor(besti, d);
        if (ob > best || (ob == best && oi < besti)) { best = ob; besti = oi; }
    }
    __syncthreads();
    if (lane == 0) { fred[wave] = best; ired[wave] = besti; }
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < 16; ++w)
            if (fred[w] > best || (fred[w] == best && ired[w] < besti)) { best = fred[w]; besti = ired[w]; }
        besti = besti < V ? besti : 0;  // (a row of NaNs)
        token_out[row] = besti;
        const unsigned long long c = rng[2 * row + 1];
        if (history && c < (unsigned long long)history_len) history[(size_t)row * history_len + c] = besti;
        rng[2 * row + 1] = c + 1ull;
        if (pos_inout) pos_inout[row] += 1;
    }
}

}  // namespace teal

using namespace teal;

extern "C" {

static int resid_norm_launch(const ResidNormArgs& a, int n_rows, int dtype, void* stream) {
    const bool y = a.y != nullptr;
    if (!a.x || n_rows <= 0 || a.D <= 0 || (a.tokens && (!a.embed || a.vocab <= 0)) || (a.post_w && !y) || (a.y_bias && !y) || (a.pre_w && !a.h)) return TEAL_ERR_ARG;
    if (a.D > 15360 || (y && a.ldy < a.D)) return TEAL_ERR_SHAPE;
    if (!device_ctx()) return TEAL_ERR_NO_DEVICE;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const void* ps[] = {a.x, a.embed, a.y, a.y_bias, a.post_w, a.pre_w, a.h};
    bool vec = (a.D & 3) == 0 && (!y || (a.ldy & 3) == 0);
    for (const void* p : ps) vec = vec && aligned16(p);
    return with_dtype(dtype, [&](auto dt) {
        constexpr int DT = decltype(dt)::value;
        const size_t lds = (size_t)a.D * sizeof(float);
#define TEAL_RN(NT, V) hipLaunchKernelGGL((resid_norm_kernel<DT, NT, V>), dim3(n_rows), dim3(NT), lds, st, a)
        if (!vec) TEAL_RN(256, 1);
        else if (a.D <= 2048) TEAL_RN(256, 4);
        else TEAL_RN(1024, 4);
#undef TEAL_RN
        return launched();
    });
}

int teal_layer_resid_norm(float* x, int n_rows, int dim, const int32_t* tokens, const void* embed, int vocab, const void* y, int ldy,
                          const void* y_bias, const void* post_w, const void* pre_w, float norm_offset, float eps, void* h, const int32_t* rows, int dtype,
                          void* stream) {
    return resid_norm_launch({x, tokens, embed, y, y_bias, post_w, pre_w, h, rows, dim, ldy, vocab, eps, norm_offset, 0, 0, nullptr, 0}, n_rows, dtype, stream);
}

int teal_layer_resid_norm_slabs(float* x, int n_rows, int dim, const int32_t* tokens, const void* embed, int vocab, const float* y, int n_slabs, int slab_rows,
                                int ldy, const void* y_bias, const void* post_w, const void* pre_w, float norm_offset, float eps, void* h,
                                const int32_t* rows, unsigned* zero, int n_zero, int dtype, void* stream) {
    if ((y && (n_slabs < 1 || slab_rows < 1)) || (zero && (n_zero < 1 || n_zero > 256))) return TEAL_ERR_ARG;
    return resid_norm_launch({x, tokens, embed, y, y_bias, post_w, pre_w, h, rows, dim, ldy, vocab, eps, norm_offset, y ? n_slabs : 0, slab_rows, zero, zero ? n_zero : 0},
                             n_rows, dtype, stream);
}

int teal_gated_act(const void* gu, int ldg, int up0, const void* bias_gate, const void* bias_up, void* h, int ldh, int n_rows, int n_cols, int act,
                   int dtype, void* stream) {
    if (!gu || !h || n_rows <= 0 || n_cols <= 0 || (act != TEAL_ACT_SILU && act != TEAL_ACT_GELU_TANH && act != TEAL_ACT_RELU2)) return TEAL_ERR_ARG;
    if (ldg < up0 + n_cols || (up0 != 0 && up0 < n_cols) || ldh < n_cols || (up0 == 0 && bias_up)) return TEAL_ERR_SHAPE;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    const bool vec = !(ldg & 7) && !(up0 & 7) && !(ldh & 7) && aligned16(gu) && aligned16(h) && aligned16(bias_gate) && aligned16(bias_up);
    return with_dtype(dtype, [&](auto dt) {
        constexpr int DT = decltype(dt)::value;
        using S = typename Num<DT>::S;
        hipLaunchKernelGGL((gated_act_kernel<DT>), dim3(n_rows, (n_cols + 2047) / 2048), dim3(256), 0, st, reinterpret_cast<const S*>(gu), ldg, up0,
                           reinterpret_cast<const S*>(bias_gate), reinterpret_cast<const S*>(bias_up), reinterpret_cast<S*>(h), ldh, n_cols, act, vec);
        return launched();
    });
}

int teal_logit_softcap(const void* logits, int ld, float* out, int n_rows, int vocab, float cap, int dtype, void* stream) {
    if (!logits || !out || n_rows <= 0 || vocab <= 0) return TEAL_ERR_ARG;
    if (ld < vocab) return TEAL_ERR_SHAPE;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    return with_dtype(dtype, [&](auto dt) {
        constexpr int DT = decltype(dt)::value;
        hipLaunchKernelGGL((softcap_kernel<DT>), dim3(n_rows, (vocab + 255) / 256), dim3(256), 0, st,
                           reinterpret_cast<const typename Num<DT>::S*>(logits), ld, out, vocab, cap);
        return launched();
    });
}

int teal_sample_rows(const float* logits, int ld, int n_rows, int vocab, int top_k, float temperature, void* rng_state, int32_t* token_out, int32_t* pos_inout,
                     int32_t* history, int history_len, void* stream) {
    if (!logits || !rng_state || !token_out || n_rows <= 0 || vocab <= 0 || (history && history_len <= 0)) return TEAL_ERR_ARG;
    if (ld < vocab) return TEAL_ERR_SHAPE;
    const bool vec = !(vocab & 3) && !(ld & 3) && aligned16(logits);
#define TEAL_SR(P) hipLaunchKernelGGL((sample_rows_kernel<P>), dim3(n_rows), dim3(1024), 0, reinterpret_cast<hipStream_t>(stream), logits, ld, vocab, top_k, \
                       temperature > 0.0f ? 1.0f / temperature : 0.0f, reinterpret_cast<unsigned long long*>(rng_state), token_out, pos_inout, history, history_len)
    if (vec && vocab <= 4096 * 2) TEAL_SR(2);
    else if (vec && vocab <= 4096 * 8) TEAL_SR(8);
    else TEAL_SR(0);
#undef TEAL_SR
    return launched();
}

}  // extern "C"
