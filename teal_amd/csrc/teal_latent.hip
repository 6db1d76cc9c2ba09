// teal_latent.hip — latent attention (one low-rank latent per token shared by all heads, plus one rotated key part) for
// gfx950 / CDNA4, wave64.  Per token and layer the cache holds ONE row [c (rank) | rotated key part (rot)], padded to a multiple
// of 32 elements; pages of 2^shift rows, a page table per sequence slot.
//
//   score(p, j, head) = (q_head . k_head(j) + rotate(qr_head, p) . kr(j)) * scale,   k_head = W_uk,head c,  v_head = W_uv,head c
//   weights: softmax over the keys p - window < j <= p, optionally with exp(sink_head) in the denominator
//   y_head = (sum_j weight_j v_head(j)) [* sigmoid(gate_head)]
//
// Prompts run in the EXPANDED form (keys and values of every head from two matrix products over the packed latents, then a flash
// attention over matrix-core tiles); single tokens run in the ABSORBED form: W_uk moves to the query side (q_abs = W_uk^T q, one
// vector of the latent's size per head), the attention works on the cached rows themselves — each row is read once for sixteen
// heads — and W_uv is applied to the weighted latent.
//
// Precision: scores, softmax weights and sums are fp32.  Where fp32 values meet the 16-bit matrix cores (the absorbed query, the
// softmax weights) they are carried as a high and a low 16-bit half and multiplied twice: the products see ~16 bits of mantissa.
// With 32-bit elements the scalar kernels run instead: plain fp32 multiply-adds.
//
// The attention kernels themselves (prompt_attention_*, step_attention_*) also serve grouped-query attention (teal_grouped.hip): `group`
// query heads share a key / value head (prompts) or a segment of the cached row (single tokens), and scores can be soft-capped.
#include "teal_rows_core.h"

namespace teal {

constexpr int kMaxStepSplits = 64;  // workgroups a sequence's cached rows may be split over
constexpr int kStepKSteps = 20;  // 32-wide inner-dimension steps of the absorbed score product: cached rows of up to 640 elements

// ------------------------------------------------------------------------------------------------
// Prompt pass, part 1: one workgroup per token.  Rotates the queries' rotated parts in place and, for a layer that owns its
// latents, writes the token's cache row: RMSNorm(latent) * w and the rotated shared key part.
// ------------------------------------------------------------------------------------------------
struct LatentRowArgs {
    void* proj;            // [T][ldp]: q at column 0 (heads x (dim + rot)), the latent and the shared key part at column kv0
    const int32_t* pos;    // [T]
    const int32_t* row;    // [T] cache row (or null with kv0 < 0)
    const float* inv_freq; // [rot / 2]
    const void* norm_w;    // [rank]
    void* cache;           // [rows][ldc]
    int ldp, kv0, heads, dim, rot, rank, ldc;
    float eps;
};

template <int DT>
__device__ __forceinline__ void latent_row(const LatentRowArgs& a, const typename Num<DT>::S* __restrict__ kv, const int p,
                                           typename Num<DT>::S* __restrict__ out, float* red, const int tid) {
    using N = Num<DT>;
    float ss = 0.0f;
    for (int i = tid; i < a.rank; i += 256) {
        const float v = N::ld(kv + i);
        ss = fmaf(v, v, ss);
    }
    const float rstd = 1.0f / sqrtf(block_sum<256>(ss, red, tid) / (float)a.rank + a.eps);
    const typename N::S* w = reinterpret_cast<const typename N::S*>(a.norm_w);
    for (int i = tid; i < a.rank; i += 256) out[i] = N::cvt(N::ld(kv + i) * rstd * N::ld(w + i));
    for (int i = tid; i < a.rot / 2; i += 256) {
        float x, y;
        rotate_pair(N::ld(kv + a.rank + 2 * i), N::ld(kv + a.rank + 2 * i + 1), p, a.inv_freq[i], x, y);
        out[a.rank + 2 * i] = N::cvt(x);
        out[a.rank + 2 * i + 1] = N::cvt(y);
    }
    for (int i = a.rank + a.rot + tid; i < a.ldc; i += 256) out[i] = (typename N::S)0;  // (the step's score product runs over whole rows)
}

template <int DT>
__global__ __launch_bounds__(256) void latent_prompt_rows_kernel(const LatentRowArgs a) {
    using N = Num<DT>;
    using S = typename N::S;
    __shared__ float red[4];
    const int tid = threadIdx.x, p = a.pos[blockIdx.x], half = a.rot / 2;
    S* proj = reinterpret_cast<S*>(a.proj) + (size_t)blockIdx.x * a.ldp;
    for (int i = tid; i < a.heads * half; i += 256) {
        const int h = i / half, j = i - h * half;
        S* q = proj + h * (a.dim + a.rot) + a.dim + 2 * j;
        float x, y;
        rotate_pair(N::ld(q), N::ld(q + 1), p, a.inv_freq[j], x, y);
        q[0] = N::cvt(x);
        q[1] = N::cvt(y);
    }
    if (a.kv0 >= 0) latent_row<DT>(a, proj + a.kv0, p, reinterpret_cast<S*>(a.cache) + (size_t)a.row[blockIdx.x] * a.ldc, red, tid);
}

// Prompt pass, part 2: the cache rows the prompt's queries can see, packed (row < 0: zeros) for the matrix products that expand them
template <int DT>
__global__ __launch_bounds__(64) void latent_gather_kernel(const typename Num<DT>::S* __restrict__ cache, const int ldc, const int32_t* __restrict__ row,
                                                           const int rank, const int rot, typename Num<DT>::S* __restrict__ c, typename Num<DT>::S* __restrict__ kr) {
    const int r = row[blockIdx.x];
    const typename Num<DT>::S* src = cache + (size_t)max(r, 0) * ldc;
    for (int i = threadIdx.x; i < rank + rot; i += 64) {
        const typename Num<DT>::S v = r >= 0 ? src[i] : (typename Num<DT>::S)0;
        if (i < rank) c[(size_t)blockIdx.x * rank + i] = v;
        else kr[(size_t)blockIdx.x * rot + i - rank] = v;
    }
}

// The same attention without the matrix cores: 32-bit elements, or head sizes beyond the tiles.  One workgroup per (query, head).
template <int DT>
__global__ __launch_bounds__(256) void prompt_attention_scalar_kernel(const PromptAttentionArgs a) {
    using N = Num<DT>;
    using S = typename N::S;
    extern __shared__ __align__(16) unsigned char smem[];
    float* q = reinterpret_cast<float*>(smem);  // [dim + rot]
    float* p = q + a.dim + a.rot;               // [256] weights of a chunk of keys
    float* part = p + 256;                      // [256] partial sums
    __shared__ float red[4];
    const int tid = threadIdx.x, head = blockIdx.y, dq = a.dim + a.rot;
    const SeqSpan sq = a.seqs[a.tiles[2 * blockIdx.x]];
    const int qi = a.tiles[2 * blockIdx.x + 1], pos = sq.start + qi;
    const S* src = reinterpret_cast<const S*>(a.q) + (size_t)(sq.q0 + qi) * a.ldq + head * dq;
    for (int i = tid; i < dq; i += 256) q[i] = N::ld(src + i);
    __syncthreads();
    const S* kp = reinterpret_cast<const S*>(a.k);
    const S* krp = reinterpret_cast<const S*>(a.kr);
    const int kvh = head / a.group, kvs = a.heads / a.group * a.dim;
    const S* vp = reinterpret_cast<const S*>(a.vt) + (size_t)kvh * a.vdim * a.S;
    const int first = max(sq.klo, pos - a.window + 1);
    // pass 1: the largest score; pass 2: weights, their sum and the weighted values (scores are computed twice, nothing is rescaled)
    auto score = [&](const int j) {
        const size_t row = (size_t)(sq.k0 + j - sq.klo);
        float s = 0.0f;
        const S* k = kp + row * kvs + kvh * a.dim;
        for (int d = 0; d < a.dim; ++d) s = fmaf(q[d], N::ld(k + d), s);
        for (int d = 0; d < a.rot; ++d) s = fmaf(q[a.dim + d], N::ld(krp + row * a.rot + d), s);
        s *= a.scale;
        return a.softcap > 0.0f ? a.softcap * tanhf(s / a.softcap) : s;
    };
    const float sink = a.sink ? N::ld(reinterpret_cast<const S*>(a.sink) + head) : -INFINITY;
    float mx = sink;
    for (int j = first + tid; j <= pos; j += 256) mx = fmaxf(mx, score(j));
    mx = block_max<256>(mx, red, tid);
    float ls = 0.0f;
    // thread (v, part): value column v of this round, one of the parts that share the keys of a chunk
    const int rounds = (a.vdim + 255) / 256;
    const int cols = min(a.vdim, 256), parts = 256 / cols;
    for (int r = 0; r < rounds; ++r) {
        const int v = r * 256 + tid % cols, pt = tid / cols;
        float acc = 0.0f;
        for (int j0 = first; j0 <= pos; j0 += 256) {
            const int j = j0 + tid;
            const float w = j <= pos ? expf(score(j) - mx) : 0.0f;
            if (r == 0) ls += w;
            __syncthreads();
            p[tid] = w;
            __syncthreads();
            if (pt < parts && v < a.vdim)
                for (int i = pt; i < min(256, pos - j0 + 1); i += parts) acc = fmaf(p[i], N::ld(vp + (size_t)v * a.S + sq.k0 + j0 + i - sq.klo), acc);
        }
        if (r == 0) ls = block_sum<256>(ls, red, tid) + (a.sink ? expf(sink - mx) : 0.0f);
        __syncthreads();
        part[tid] = acc;
        __syncthreads();
        if (tid < cols && v < a.vdim) {
            float t = 0.0f;
            for (int i = 0; i < parts; ++i) t += part[i * cols + tid];
            const size_t tok = (size_t)(sq.q0 + qi);
            t /= ls;
            if (a.gate) t *= sigmoid_f(N::ld(reinterpret_cast<const S*>(a.gate) + tok * a.ldg + head * a.vdim + v));
            reinterpret_cast<S*>(a.out)[tok * a.ldo + head * a.vdim + v] = N::cvt(t);
        }
    }
}

// ------------------------------------------------------------------------------------------------
// Single tokens, part 1: grid (heads * chunks [+ 1], batch / BT).  Workgroup (head, chunk): 128 columns of the absorbed query
// W_uk,head^T q of BT tokens (chunk 0 also rotates the query's rotated part); the extra workgroup: the tokens' cache rows.
// qcat [batch][heads][ldq]: q_abs (rank), rotated part (rot), zeros up to ldq — one fp32 row, or a high and a low 16-bit row.
// ------------------------------------------------------------------------------------------------
struct LatentStepArgs {
    LatentRowArgs kv;        // proj = [batch][ldp]; pos per batch entry; cache of the layer (kv0 < 0: another layer's, untouched)
    const int32_t* slot;     // [batch] page-table row
    const int32_t* table;    // [slots][max_pages]
    const void* uk;          // [heads * dim][rank]
    void* qcat;
    int max_pages, shift, chunks, ldq;
};

template <int DT, int BT>
__global__ __launch_bounds__(256) void latent_step_query_kernel(const LatentStepArgs a, const int batch) {
    using N = Num<DT>;
    using S = typename N::S;
    extern __shared__ __align__(16) unsigned char smem[];
    float* q = reinterpret_cast<float*>(smem);  // [BT][dim]
    __shared__ float red[4], part[16][129];
    const LatentRowArgs& k = a.kv;
    const int tid = threadIdx.x, b0 = blockIdx.y * BT, nb = min(BT, batch - b0);
    const S* proj = reinterpret_cast<const S*>(k.proj) + (size_t)b0 * k.ldp;
    if ((int)blockIdx.x == k.heads * a.chunks) {
        for (int i = 0; i < nb; ++i) {
            const int p = k.pos[b0 + i];
            const int row = page_row(a.table + (size_t)a.slot[b0 + i] * a.max_pages, min(p, (a.max_pages << a.shift) - 1), a.shift);
            latent_row<DT>(k, proj + (size_t)i * k.ldp + k.kv0, p, reinterpret_cast<S*>(k.cache) + (size_t)row * k.ldc, red, tid);
        }
        return;
    }
    const int head = blockIdx.x / a.chunks, r0 = (blockIdx.x % a.chunks) * 128;
    const S* qh = proj + head * (k.dim + k.rot);
    const int c0 = (tid & 15) * 8, dg = tid >> 4;
    const S* w = reinterpret_cast<const S*>(a.uk) + (size_t)head * k.dim * k.rank + r0 + c0;
    float acc[BT][8];
#pragma unroll
    for (int t = 0; t < BT; ++t)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[t][j] = 0.0f;
    const int left = k.rank - r0 - c0;
    const bool vec = !(k.rank & 7);
    constexpr int U = DT == TEAL_F32 ? 4 : 8;  // weight rows in flight; the first ones leave before the query has arrived
    Raw8<DT> v[U];
    auto rows = [&](const int d0) {
#pragma unroll
        for (int u = 0; u < U; ++u) v[u].load(w + (size_t)min(d0 + 16 * u, k.dim - 1) * k.rank, vec);
    };
    if (left >= 8) rows(dg);
    for (int i = tid; i < BT * k.dim; i += 256) {
        const int t = BT == 1 ? 0 : i / k.dim, d = i - t * k.dim;
        q[i] = t < nb ? N::ld(qh + (size_t)t * k.ldp + d) : 0.0f;
    }
    __syncthreads();
    if (left >= 8) {
        for (int d0 = dg; d0 < k.dim; d0 += 16 * U) {
            if (d0 != dg) rows(d0);
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int d = min(d0 + 16 * u, k.dim - 1);
                float x[BT];
#pragma unroll
                for (int t = 0; t < BT; ++t) x[t] = d0 + 16 * u < k.dim ? q[t * k.dim + d] : 0.0f;
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const float wj = v[u].get(j);
#pragma unroll
                    for (int t = 0; t < BT; ++t) acc[t][j] = fmaf(x[t], wj, acc[t][j]);
                }
            }
        }
    } else if (left > 0) {
        for (int d = dg; d < k.dim; d += 16)
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (j < left) {
                    const float wj = N::ld(w + (size_t)d * k.rank + j);
#pragma unroll
                    for (int t = 0; t < BT; ++t) acc[t][j] = fmaf(q[t * k.dim + d], wj, acc[t][j]);
                }
    }
#pragma unroll
    for (int t = 0; t < BT; ++t) {
        if (t >= nb) break;
        auto put = [&](const int i, const float x) {  // element i of this head's row
            const size_t at = (size_t)(b0 + t) * k.heads + head;
            if constexpr (DT == TEAL_F32) {
                reinterpret_cast<float*>(a.qcat)[at * a.ldq + i] = x;
            } else {
                uint32_t hi, lo;
                split16<DT == TEAL_BF16>(x, hi, lo);
                reinterpret_cast<uint16_t*>(a.qcat)[at * 2 * a.ldq + i] = (uint16_t)hi;
                reinterpret_cast<uint16_t*>(a.qcat)[(at * 2 + 1) * a.ldq + i] = (uint16_t)lo;
            }
        };
        if (t) __syncthreads();
#pragma unroll
        for (int j = 0; j < 8; ++j) part[dg][c0 + j] = acc[t][j];
        __syncthreads();
        if (tid < 128 && r0 + tid < k.rank) {
            float x = 0.0f;
#pragma unroll
            for (int i = 0; i < 16; ++i) x += part[i][tid];
            put(r0 + tid, x);
        }
        if (r0 == 0) {
            const S* qr = qh + (size_t)t * k.ldp + k.dim;
            const int p = k.pos[b0 + t];
            for (int i = tid; i < k.rot / 2; i += 256) {
                float x, y;
                rotate_pair(N::ld(qr + 2 * i), N::ld(qr + 2 * i + 1), p, k.inv_freq[i], x, y);
                put(k.rank + 2 * i, x);
                put(k.rank + 2 * i + 1, y);
            }
            for (int i = k.rank + k.rot + tid; i < a.ldq; i += 256) put(i, 0.0f);
        }
    }
}

// The same on the matrix cores, for up to sixteen tokens at once (their queries are 16-bit values: exact operands).  grid (heads * chunks
// [+ 16 tokens' cache rows], batch / 16), four waves; a wave: 64 columns of the absorbed query, W_uk straight to its registers
// (teal_rows_core.h), nothing shared.  Bound by latency: every load of 128 inputs is in flight at once.  16 tokens, 32 heads of 128, rank
// 512: 7.6 -> 4.6 us (12 -> 5 with the cache rows, which one workgroup wrote for four tokens); 64 tokens: 19.6 -> 6.8
template <bool BF16>
__global__ __launch_bounds__(256) void latent_step_query_rows_kernel(const LatentStepArgs a, const int batch) {
    constexpr int DT = BF16 ? TEAL_BF16 : TEAL_F16, FLIGHT = 4;
    __shared__ float red[4];
    const LatentRowArgs& k = a.kv;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, g = lane >> 4;
    const int b0 = blockIdx.y * 16, nb = min(16, batch - b0);
    const uint16_t* proj = reinterpret_cast<const uint16_t*>(k.proj) + (size_t)b0 * k.ldp;
    const int extra = (int)blockIdx.x - k.heads * a.chunks;
    if (extra >= 0) {
        if (extra >= nb) return;
        const int p = k.pos[b0 + extra];
        const int row = page_row(a.table + (size_t)a.slot[b0 + extra] * a.max_pages, min(p, (a.max_pages << a.shift) - 1), a.shift);
        latent_row<DT>(k, proj + (size_t)extra * k.ldp + k.kv0, p, reinterpret_cast<uint16_t*>(k.cache) + (size_t)row * k.ldc, red, tid);
        return;
    }
    const int head = blockIdx.x / a.chunks, r0 = (blockIdx.x % a.chunks) * 256;
    const uint16_t* qh = proj + head * (k.dim + k.rot);
    uint16_t* out = reinterpret_cast<uint16_t*>(a.qcat) + ((size_t)b0 * k.heads + head) * 2 * a.ldq;  // token t: + t * heads * 2 * ldq
    const int col = r0 + 64 * wave, wide = min(64, k.rank - col), ldb = 2 * k.rank, steps = k.dim / 32;
    if (wide > 0) {
        const RowsBuf buf[1] = {rows_buffer(reinterpret_cast<const uint16_t*>(a.uk) + (size_t)head * k.dim * k.rank + col, (size_t)(k.dim - 1) * ldb + 2 * wide)};
        const uint32_t base = (uint32_t)(8 * g) * (uint32_t)ldb + 8u * (uint32_t)l16;
        auto off = [&](const int s) { return 4 * l16 < wide && s < steps ? base + (uint32_t)s * 32u * (uint32_t)ldb : kRowsNowhere; };
        const uint16_t* x = qh + (size_t)min(l16, nb - 1) * k.ldp + 8 * g;
        RowsTile<4, 1> t[FLIGHT];
        u32x4 xs[FLIGHT][1];
        auto fetch = [&](const int i, const int s) {
            rows_load<4, 1>(t[i], buf, off(s), ldb);
            xs[i][0] = *reinterpret_cast<const u32x4*>(x + 32 * min(s, steps - 1));
        };
#pragma unroll
        for (int i = 0; i < FLIGHT; ++i) fetch(i, i);
        f32x4 acc[1][4];
#pragma unroll
        for (int f = 0; f < 4; ++f) acc[0][f] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int s = 0; s < steps; s += FLIGHT)
#pragma unroll
            for (int i = 0; i < FLIGHT; ++i) {  // (steps past the last: zeros of W_uk)
                rows_mfma<BF16, false, 1, 4, 1>(t[i], xs[i], acc);
                if (s + FLIGHT < steps) fetch(i, s + FLIGHT + i);
            }
        // a lane holds token l16 and the columns 16 g .. 16 g + 15 of the wave's 64
        if (l16 < nb && 16 * g < wide) {
            uint16_t* o = out + (size_t)l16 * k.heads * 2 * a.ldq + col + 16 * g;
            uint32_t hi[8], lo[8];
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int f = 0; f < 4; f += 2) split16x2<BF16>(acc[0][f][i], acc[0][f + 1][i], hi[2 * i + f / 2], lo[2 * i + f / 2]);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                *reinterpret_cast<u32x4*>(o + 8 * h) = u32x4{hi[4 * h], hi[4 * h + 1], hi[4 * h + 2], hi[4 * h + 3]};
                *reinterpret_cast<u32x4*>(o + a.ldq + 8 * h) = u32x4{lo[4 * h], lo[4 * h + 1], lo[4 * h + 2], lo[4 * h + 3]};
            }
        }
    }
    if (r0 != 0) return;
    // the rotated part and the zeros behind it
    const int pairs = k.rot / 2, tail = a.ldq - k.rank - k.rot, per = pairs + tail;
    for (int i = tid; i < nb * per; i += 256) {
        const int t = i / per, j = i - t * per;
        uint16_t* o = out + (size_t)t * k.heads * 2 * a.ldq;
        if (j >= pairs) {
            const int c = k.rank + k.rot + j - pairs;
            o[c] = o[a.ldq + c] = 0;
            continue;
        }
        const uint16_t* qr = qh + (size_t)t * k.ldp + k.dim + 2 * j;
        float v[2];
        rotate_pair(bits_to_float(qr[0], BF16), bits_to_float(qr[1], BF16), k.pos[b0 + t], k.inv_freq[j], v[0], v[1]);
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            uint32_t hi, lo;
            split16<BF16>(v[e], hi, lo);
            o[k.rank + 2 * j + e] = (uint16_t)hi;
            o[a.ldq + k.rank + 2 * j + e] = (uint16_t)lo;
        }
    }
}

// ------------------------------------------------------------------------------------------------
// Single tokens, part 2: attention over the cached rows.  grid (splits, groups of up to 16 heads of one segment, batch), four waves.  A split takes a run of
// 32-key tiles of the window.  Per tile: the waves share the score product by its inner dimension (both 16-key tiles, K steps
// wave, wave + 4, ...; partial scores through LDS), then each wave owns a quarter of the latent's columns in the value product.
// A tile's rows are read once, into the LDS as they lie: the score product takes eight elements of a row, the value product four rows of a
// column (ds_read_b64_tr_b16); the next tile is on its way meanwhile.  Bound by what one CU can load: fetched twice, as operands and to be
// stored transposed, 16 tokens of 32 heads at 1000 positions took 18.2 us, 14.0 now;
// one token 7.4 and 6.0.
// part [batch][heads][splits][part_stride(rank)] = {weighted latent (rank, padded to 4), max (log2 units), sum, -, -}.
// ------------------------------------------------------------------------------------------------
__host__ __device__ constexpr int part_stride(const int rank) { return ((rank + 3) & ~3) + 4; }

struct StepAttentionArgs {
    const void* qcat;
    const void* cache;
    const int32_t* pos;
    const int32_t* slot;
    const int32_t* table;
    float* part;
    int max_pages, shift, ldq, ldc, heads, group, rank, rot, window, splits;  // a cached row (ldc) holds heads / group segments of ldq elements
    float scale, softcap;
    // TIED instantiations: the projection's rows (queries at column 0, keys at k0) and the rotation; the kernel makes its query rows and the
    // token's cache row itself
    const void* proj;
    const float* inv_freq;
    int ldp, k0;
};

struct KeyRange { int lo, hi; };  // first position, one past the last

// the share of [max(0, p - window + 1), p] a split takes: whole tiles of `tile` keys, aligned in position
__device__ __forceinline__ KeyRange split_range(const int p, const int window, const int split, const int splits, const int tile) {
    const int lo = max(0, p - window + 1);
    const int t0 = lo / tile, nt = p / tile - t0 + 1;
    const int per = (nt + splits - 1) / splits;
    KeyRange r;
    r.lo = max(lo, (t0 + split * per) * tile);
    r.hi = min(p + 1, (t0 + (split + 1) * per) * tile);
    return r;
}

// elements between the rows of a tile in the LDS: whole tiles of value columns, and 16 bytes more so that rows start in different banks
__host__ __device__ inline int step_tile_row(const int ldq, const int rt) { return (ldq > rt * 16 ? ldq : rt * 16) + 8; }

// TIED: the workgroups that hold the token's own key write its cache row before they read it (several of them, more than sixteen heads
// to a key head: the same values).
template <bool BF16, int RT, bool TIED, bool CAPPED>
__global__ __launch_bounds__(256) void step_attention_kernel(const StepAttentionArgs a) {
    constexpr int RPW = RT / 4, KSW = kStepKSteps / 4, NI = kStepKSteps / 2;  // 16-column tiles, inner-dimension steps per wave; pieces of a row per thread
    __shared__ __align__(16) float sp[4 * 2 * 64 * 4];  // partial scores, lane-major
    extern __shared__ __align__(16) unsigned char dyn[];
    uint16_t* ct = reinterpret_cast<uint16_t*>(dyn);    // [32 keys][LD]
    const int LD = step_tile_row(a.ldq, RT);
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, g = lane >> 4;
    const int per = (a.group + 15) / 16, seg = blockIdx.y / per;
    const int split = blockIdx.x, h0 = seg * a.group + (blockIdx.y - seg * per) * 16, b = blockIdx.z;
    const int nh = min(16, (seg + 1) * a.group - h0);
    const int p = min(a.pos[b], (a.max_pages << a.shift) - 1);  // (a position past the table would read past it)
    const int* table = a.table + (size_t)a.slot[b] * a.max_pages;
    const int ksteps = a.ldq / 32;
    const KeyRange kr = split_range(p, a.window, split, a.splits, 32);
    if (TIED && kr.lo >= kr.hi) {  // (nothing of the window is left for this split)
        if (tid < nh) {
            const int r4 = part_stride(a.rank) - 4;
            float* out = a.part + (((size_t)b * a.heads + h0 + tid) * a.splits + split) * (r4 + 4);
            out[r4] = -INFINITY;
            out[r4 + 1] = 0.0f;
        }
        return;
    }
    if constexpr (TIED) {
        constexpr int DT = BF16 ? TEAL_BF16 : TEAL_F16;
        uint16_t* qs = reinterpret_cast<uint16_t*>(dyn);  // [nh][2][ldq], where the first tile comes to lie later
        const uint16_t* proj = reinterpret_cast<const uint16_t*>(a.proj) + (size_t)b * a.ldp;
        for (int i = tid; i < nh * a.ldq; i += 256) {
            const int h = i / a.ldq, d = i - h * a.ldq;
            uint32_t hi, lo;
            split16<BF16>(tied_query_element<DT>(proj + (size_t)(h0 + h) * a.rank, d, a.rank, a.rot, p, a.inv_freq), hi, lo);
            qs[2 * h * a.ldq + d] = (uint16_t)hi;
            qs[(2 * h + 1) * a.ldq + d] = (uint16_t)lo;
        }
        if (kr.hi == p + 1) {
            uint16_t* out = reinterpret_cast<uint16_t*>(const_cast<void*>(a.cache)) + (size_t)page_row(table, p, a.shift) * a.ldc + (size_t)seg * a.ldq;
            for (int d = tid; d < a.ldq; d += 256) out[d] = tied_row_element<DT>(proj + a.k0 + (size_t)seg * a.rank, d, a.rank, a.rot, p, a.inv_freq);
        }
        __threadfence_block();
        __syncthreads();
    }
    // this wave's part of the query rows, high and low halves: operand rows of sixteen heads
    u32x4 qf[KSW][2];
    {
        const int row = min(l16, nh - 1);
        const uint16_t* q = TIED ? reinterpret_cast<const uint16_t*>(dyn) + (size_t)row * 2 * a.ldq + g * 8
                                 : reinterpret_cast<const uint16_t*>(a.qcat) + ((size_t)b * a.heads + h0 + row) * 2 * a.ldq + g * 8;
#pragma unroll
        for (int s = 0; s < KSW; ++s)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                qf[s][h] = u32x4{0u, 0u, 0u, 0u};
                if (wave + 4 * s < ksteps) qf[s][h] = *reinterpret_cast<const u32x4*>(q + h * a.ldq + (wave + 4 * s) * 32);
            }
    }
    const uint16_t* cache = reinterpret_cast<const uint16_t*>(a.cache) + (size_t)seg * a.ldq;
    const float sc = score_factor<CAPPED>(a.scale, a.softcap), cl2 = a.softcap * kLog2e;
    float m = -INFINITY, l = 0.0f;
    f32x4 o[RPW];
#pragma unroll
    for (int r = 0; r < RPW; ++r) o[r] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (TIED) __syncthreads();  // (every wave has its queries)
    // a thread's pieces: 16 bytes of row tid / 8, every eighth of the row.  Keys outside the share read as zeros (their rows may be another
    // sequence's leftovers): they are requested outside the buffer
    const int krow = tid >> 3, kc = tid & 7, ni = (a.ldq + 63) / 64;
    u32x4 st[NI];
    auto fetch = [&](const int j0, const int base) {
        const RowsBuf buf = rows_buffer(cache + (size_t)base * a.ldc, ((size_t)31 * a.ldc + a.ldq) * 2);
        const uint32_t off = j0 + krow >= kr.lo && j0 + krow < kr.hi ? (uint32_t)krow * (uint32_t)(2 * a.ldc) + 16u * (uint32_t)kc : kRowsNowhere;
#pragma unroll
        for (int i = 0; i < NI; ++i)
            if (i < ni) st[i] = __builtin_amdgcn_raw_buffer_load_b128(buf, (int)(8 * (kc + 8 * i) < a.ldq ? off + (off == kRowsNowhere ? 0u : 128u * i) : kRowsNowhere), 0, 0);
    };
    auto lds_barrier = [&]() {  // (not __syncthreads(), which would wait for the next tile as well)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    const int jend = (kr.hi - 1) / 32 * 32;  // (a tile of 32 keys never crosses a page: pages hold 2^shift >= 32)
    int j0 = kr.lo / 32 * 32;
    int next = 0;
    if (kr.lo < kr.hi) {
        fetch(j0, page_row(table, j0, a.shift));
        next = page_row(table, min(j0 + 32, jend), a.shift);
    }
    for (; j0 < kr.hi && kr.lo < kr.hi; j0 += 32) {
#pragma unroll
        for (int i = 0; i < NI; ++i)
            if (i < ni && 8 * (kc + 8 * i) < a.ldq) *reinterpret_cast<u32x4*>(ct + krow * LD + 8 * (kc + 8 * i)) = st[i];
        lds_barrier();
        f32x4 s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int q = 0; q < KSW; ++q)
            if (wave + 4 * q < ksteps) {
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const u32x4 kf = *reinterpret_cast<const u32x4*>(ct + (t * 16 + l16) * LD + (wave + 4 * q) * 32 + 8 * g);
                    s[t] = mfma16<BF16>(kf, qf[q][0], s[t]);
                    s[t] = mfma16<BF16>(kf, qf[q][1], s[t]);
                }
            }
#pragma unroll
        for (int t = 0; t < 2; ++t) *reinterpret_cast<f32x4*>(sp + ((wave * 2 + t) * 64 + lane) * 4) = s[t];
        if (j0 + 32 < kr.hi) {
            const int base = next;
            next = page_row(table, min(j0 + 64, jend), a.shift);
            fetch(j0 + 32, base);
        }
        lds_barrier();
        float mx = m;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int w = 0; w < 4; ++w) v += *reinterpret_cast<const f32x4*>(sp + ((w * 2 + t) * 64 + lane) * 4);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int j = j0 + t * 16 + g * 4 + r;
                const float z = CAPPED ? soft_cap2(v[r] * sc, cl2) : v[r] * sc;
                s[t][r] = (j >= kr.lo && j < kr.hi) ? z : -INFINITY;
                mx = fmaxf(mx, s[t][r]);
            }
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        const float ms = mx == -INFINITY ? 0.0f : mx;
        const float al = exp2_fast(m - ms);
        m = mx;
        u32x4 ph, pl;
        float ls = 0.0f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float p0 = exp2_fast(s[j >> 1][2 * (j & 1)] - ms), p1 = exp2_fast(s[j >> 1][2 * (j & 1) + 1] - ms);
            uint32_t hi, lo;
            split16x2<BF16>(p0, p1, hi, lo);
            ph[j] = hi;
            pl[j] = lo;
            ls += p0 + p1;
        }
        l = l * al + ls;
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
            const uint16_t* bp = ct + (g * 4 + (l16 >> 2)) * LD + (wave * RPW + r) * 16 + 4 * (l16 & 3);
            const u32x2 w0 = lds_column4(bp), w1 = lds_column4(bp + 16 * LD);
            const u32x4 cf = {w0[0], w0[1], w1[0], w1[1]};
            o[r] *= al;
            o[r] = mfma16<BF16>(cf, ph, o[r]);
            o[r] = mfma16<BF16>(cf, pl, o[r]);
        }
        lds_barrier();
    }
    l += __shfl_xor(l, 16);
    l += __shfl_xor(l, 32);
    if (l16 < nh) {
        const int r4 = part_stride(a.rank) - 4;
        float* out = a.part + (((size_t)b * a.heads + h0 + l16) * a.splits + split) * (r4 + 4);
        if (wave == 0 && g == 0) { out[r4] = m; out[r4 + 1] = l; }
#pragma unroll
        for (int r = 0; r < RPW; ++r) {
            const int c = (wave * RPW + r) * 16 + g * 4;
            if (c < r4) *reinterpret_cast<f32x4*>(out + c) = o[r];  // (columns past the rank: other parts of the rows, never read)
        }
    }
}

// The same without the matrix cores (32-bit elements, or ranks beyond the tiles): one workgroup per (split, head, batch entry)
template <int DT>
__global__ __launch_bounds__(256) void step_attention_scalar_kernel(const StepAttentionArgs a) {
    using N = Num<DT>;
    using S = typename N::S;
    extern __shared__ __align__(16) unsigned char smem[];
    const int D = a.rank + a.rot;
    float* q = reinterpret_cast<float*>(smem);  // [D]
    float* o = q + D;                           // [rank]
    __shared__ float pw[256], red[4];
    __shared__ int rows[256];
    const int tid = threadIdx.x, split = blockIdx.x, head = blockIdx.y, b = blockIdx.z;
    const int p = min(a.pos[b], (a.max_pages << a.shift) - 1);
    const int* table = a.table + (size_t)a.slot[b] * a.max_pages;
    const size_t at = (size_t)b * a.heads + head;
    for (int i = tid; i < D; i += 256) {
        if constexpr (DT == TEAL_F32) q[i] = reinterpret_cast<const float*>(a.qcat)[at * a.ldq + i];
        else q[i] = N::ld(reinterpret_cast<const S*>(a.qcat) + at * 2 * a.ldq + i) + N::ld(reinterpret_cast<const S*>(a.qcat) + (at * 2 + 1) * a.ldq + i);
        if (i < a.rank) o[i] = 0.0f;
    }
    __syncthreads();
    const KeyRange kr = split_range(p, a.window, split, a.splits, 32);
    const S* cache = reinterpret_cast<const S*>(a.cache) + (size_t)(head / a.group) * a.ldq;
    float m = -INFINITY, l = 0.0f;
    for (int j0 = kr.lo; j0 < kr.hi; j0 += 256) {
        const int j = j0 + tid, row = page_row(table, min(j, kr.hi - 1), a.shift);
        float s = 0.0f;
        const S* c = cache + (size_t)row * a.ldc;
        for (int d = 0; d < D; ++d) s = fmaf(q[d], N::ld(c + d), s);
        s *= a.scale;
        if (a.softcap > 0.0f) s = a.softcap * tanhf(s / a.softcap);
        s = j < kr.hi ? s * kLog2e : -INFINITY;
        const float mx = fmaxf(m, block_max<256>(s, red, tid));
        const float al = exp2f(m - mx), w = j < kr.hi ? exp2f(s - mx) : 0.0f;
        m = mx;
        l = l * al + block_sum<256>(w, red, tid);
        pw[tid] = w;
        rows[tid] = row;
        __syncthreads();
        const int n = min(256, kr.hi - j0);
        for (int r = tid; r < a.rank; r += 256) {
            float acc = o[r] * al;
            for (int i = 0; i < n; ++i) acc = fmaf(pw[i], N::ld(cache + (size_t)rows[i] * a.ldc + r), acc);
            o[r] = acc;
        }
        __syncthreads();
    }
    const int r4 = part_stride(a.rank) - 4;
    float* out = a.part + (at * a.splits + split) * (r4 + 4);
    if (tid == 0) { out[r4] = m; out[r4 + 1] = l; }
    for (int r = tid; r < r4; r += 256) out[r] = r < a.rank ? o[r] : 0.0f;
}

// ------------------------------------------------------------------------------------------------
// Single tokens, part 3: merge the splits (and the sink), apply W_uv and the gate.  grid (column chunks of 32, heads, batch).
// ------------------------------------------------------------------------------------------------
struct LatentMergeArgs {
    const float* part;
    const void* uv;     // [heads * vdim][rank]
    const void* sink;   // or null: [heads]
    const void* gate;   // or null: [batch][ldg], heads x vdim
    void* y;            // [batch][ldy]
    int heads, rank, vdim, splits, ldg, ldy;
};

template <int DT, int BT>
__global__ __launch_bounds__(256) void latent_decode_merge_kernel(const LatentMergeArgs a, const int batch) {
    using N = Num<DT>;
    using S = typename N::S;
    extern __shared__ __align__(16) unsigned char smem[];
    const int lo = (a.rank + 7) & ~7;
    float* o = reinterpret_cast<float*>(smem);  // [BT][rank rounded up to 8]
    float* sum = o + BT * lo;                   // [1024] partial sums of groups of splits
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, head = blockIdx.y, b0 = blockIdx.z * BT, nb = min(BT, batch - b0);
    const int stride = part_stride(a.rank), r4 = stride - 4;
    // what does not depend on the weights of the splits leaves first: this wave's eight rows of W_uv (lane: eight of the latent's
    // columns, the first 512 of them), the gate and the sink
    const int v0 = blockIdx.x * 32 + wave * 8, nv = min(8, a.vdim - v0);
    const S* w = reinterpret_cast<const S*>(a.uv) + (size_t)(head * a.vdim + min(v0, a.vdim - 1)) * a.rank;
    const bool vec = !(a.rank & 7);
    auto full = [&](const int c0) { return c0 + 8 <= a.rank && nv > 0; };
    Raw8<DT> wv[8];
    auto weights = [&](const int c0) {
#pragma unroll
        for (int i = 0; i < 8; ++i) wv[i].load(w + (size_t)min(i, nv - 1) * a.rank + c0, vec);
    };
    if (full(lane * 8)) weights(lane * 8);
    const int col = head * a.vdim + min(v0 + min(lane, 7), a.vdim - 1);  // (lanes 0 .. nv - 1: their own output column)
    float gt[BT];
#pragma unroll
    for (int t = 0; t < BT; ++t) gt[t] = a.gate ? N::ld(reinterpret_cast<const S*>(a.gate) + (size_t)(b0 + min(t, nb - 1)) * a.ldg + col) : 0.0f;
    const float sink2 = a.sink ? N::ld(reinterpret_cast<const S*>(a.sink) + head) * kLog2e : -INFINITY;
#pragma unroll 1
    for (int t = 0; t < nb; ++t) {
        const float* part = a.part + ((size_t)(b0 + t) * a.heads + head) * a.splits * stride;
        // thread: four columns of the latent, every `groups`-th split; the first eight partials leave before the factors are known
        const int quads = r4 / 4, groups = quads >= 256 ? 1 : 256 / quads;
        const int grp = quads >= 256 ? 0 : tid / quads, quad0 = quads >= 256 ? tid : tid % quads;
        const bool act = grp < groups;
        auto at = [&](const int s, const int quad) { return *reinterpret_cast<const f32x4*>(part + (size_t)min(s, a.splits - 1) * stride + 4 * quad); };
        f32x4 y[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) y[u] = at((act ? grp : 0) + groups * u, min(quad0, quads - 1));
        // every wave for itself: lane = split (kMaxStepSplits of them), no barriers
        const float pm = lane < a.splits ? part[(size_t)lane * stride + r4] : -INFINITY, pl = lane < a.splits ? part[(size_t)lane * stride + r4 + 1] : 0.0f;
        const float M = fmaxf(sink2, wave_max_f(pm));
        const float pf = lane < a.splits ? exp2f(pm - M) : 0.0f;
        const float inv = 1.0f / (wave_sum_f(pl * pf) + (a.sink ? exp2f(sink2 - M) : 0.0f));
        for (int q0 = 0; q0 < quads; q0 += 256) {  // (uniform trip counts: the factors come from other lanes)
            const int quad = min(q0 + quad0, quads - 1);
            const bool mine = act && q0 + quad0 < quads;
            f32x4 x = {0.f, 0.f, 0.f, 0.f};
            for (int s0 = 0; s0 < a.splits; s0 += 8 * groups) {
                const int s = s0 + (act ? grp : 0);
                if (s0 != 0 || q0 != 0) {
#pragma unroll
                    for (int u = 0; u < 8; ++u) y[u] = at(s + groups * u, quad);
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const float fs = __shfl(pf, min(s + groups * u, 63));
                    if (s + groups * u < a.splits) x += y[u] * fs;
                }
            }
            if (mine && groups > 1) {
                *reinterpret_cast<f32x4*>(sum + (grp * quads + quad) * 4) = x;
            } else if (mine) {
#pragma unroll
                for (int j = 0; j < 4; ++j) if (4 * quad + j < lo) o[t * lo + 4 * quad + j] = 4 * quad + j < a.rank ? x[j] * inv : 0.0f;
            }
        }
        if (groups > 1) {
            __syncthreads();  // (the next token's writes wait behind the barrier below)
            for (int r = tid; r < lo; r += 256) {
                float x = 0.0f;
                for (int g = 0; g < groups; ++g) x += r < r4 ? sum[g * r4 + r] : 0.0f;
                o[t * lo + r] = r < a.rank ? x * inv : 0.0f;
            }
            if (t + 1 < nb) __syncthreads();
        } else {
            for (int r = r4 + tid; r < lo; r += 256) o[t * lo + r] = 0.0f;
        }
    }
    __syncthreads();
    if (nv <= 0) return;
    float acc[BT][8];
#pragma unroll
    for (int t = 0; t < BT; ++t)
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[t][i] = 0.0f;
    for (int c0 = lane * 8; c0 < a.rank; c0 += 512) {
        if (full(c0)) {
            if (c0 != lane * 8) weights(c0);
#pragma unroll
            for (int t = 0; t < BT; ++t) {
                if (t >= nb) break;
                float x[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) x[j] = o[t * lo + c0 + j];
#pragma unroll
                for (int i = 0; i < 8; ++i)
#pragma unroll
                    for (int j = 0; j < 8; ++j) acc[t][i] = fmaf(wv[i].get(j), x[j], acc[t][i]);
            }
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (i < nv)
                    for (int j = c0; j < a.rank; ++j) {
                        const float x = N::ld(w + (size_t)i * a.rank + j);
#pragma unroll
                        for (int t = 0; t < BT; ++t) acc[t][i] = t < nb ? fmaf(x, o[t * lo + j], acc[t][i]) : 0.0f;
                    }
        }
    }
#pragma unroll
    for (int t = 0; t < BT; ++t) {
        if (t >= nb) break;
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[t][i] = wave_sum_f(acc[t][i]);
        float x = acc[t][0];
#pragma unroll
        for (int i = 1; i < 8; ++i) x = lane == i ? acc[t][i] : x;
        if (a.gate) x *= sigmoid_f(gt[t]);
        if (lane < nv) reinterpret_cast<S*>(a.y)[(size_t)(b0 + t) * a.ldy + col] = N::cvt(x);
    }
}

// The same on the matrix cores, four tokens to a workgroup of four waves: wave t merges token t's splits (a lane: two quads of the latent at a time,
// eight splits in flight, no barrier), leaves the merged fp32 latent as three 16-bit parts that add up to it (24 bits: as exact
// as the fp32 products above), and the product with W_uv has them as twelve rows.  A wave: 16 of the workgroup's 64 columns.  Bound by the partial results,
// which a workgroup reads for its tokens and every 64 columns of the head.  32 heads, rank 512, vdim 128: 16 tokens
// of 16 splits 17.3 -> 8.1 us, of 8 splits 14.5 -> 5.6; 64 tokens of 4 splits 49 -> 13.9
template <bool BF16>
__global__ __launch_bounds__(256) void latent_merge_rows_kernel(const LatentMergeArgs a, const int batch) {
    extern __shared__ __align__(16) unsigned char smem[];
    uint16_t* op = reinterpret_cast<uint16_t*>(smem);  // [part * 4 + token][rank + 8]
    constexpr int FLIGHT = 16;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), l16 = lane & 15, g = lane >> 4, head = blockIdx.y;
    const int b0 = blockIdx.z * 4, nb = min(4, batch - b0), lo = a.rank + 8, steps = a.rank / 32;
    const int stride = part_stride(a.rank), r4 = stride - 4, quads = a.rank / 4;
    // W_uv: rows (columns of the result) past the head's last lie outside the buffer and read as zeros
    const int v = blockIdx.x * 64 + wave * 16 + l16;
    const RowsBuf buf = rows_buffer(reinterpret_cast<const uint16_t*>(a.uv) + (size_t)head * a.vdim * a.rank, (size_t)a.vdim * a.rank * 2);
    const uint32_t base = v < a.vdim ? ((uint32_t)v * (uint32_t)a.rank + 8u * (uint32_t)g) * 2u : kRowsNowhere;
    const float sink2 = a.sink ? bits_to_float(reinterpret_cast<const uint16_t*>(a.sink)[head], BF16) * kLog2e : -INFINITY;
    const size_t vc = (size_t)head * a.vdim + min(v, a.vdim - 1);
    const float gt = a.gate ? bits_to_float(reinterpret_cast<const uint16_t*>(a.gate)[(size_t)(b0 + min(g, nb - 1)) * a.ldg + vc], BF16) : 0.0f;
    u32x4 w[FLIGHT];
    auto weights = [&](const int s0) {
#pragma unroll
        for (int i = 0; i < FLIGHT; ++i) w[i] = __builtin_amdgcn_raw_buffer_load_b128(buf, (int)(s0 + i < steps ? base + 64u * (uint32_t)(v < a.vdim ? s0 + i : 0) : kRowsNowhere), 0, 0);
    };
    if (wave < nb) {
        const float* part = a.part + ((size_t)(b0 + wave) * a.heads + head) * a.splits * stride;
        f32x4 y[8][2];
        auto load = [&](const int s0, const int q0) {
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int e = 0; e < 2; ++e) y[u][e] = *reinterpret_cast<const f32x4*>(part + (size_t)min(s0 + u, a.splits - 1) * stride + 4 * min(q0 + 64 * e + lane, quads - 1));
        };
        const float pm = lane < a.splits ? part[(size_t)lane * stride + r4] : -INFINITY, pl = lane < a.splits ? part[(size_t)lane * stride + r4 + 1] : 0.0f;
        load(0, 0);
        weights(0);
        const float M = fmaxf(sink2, wave_max_f(pm));
        const float pf = lane < a.splits ? exp2f(pm - M) : 0.0f;
        const float inv = 1.0f / (wave_sum_f(pl * pf) + (a.sink ? exp2f(sink2 - M) : 0.0f));
        for (int q0 = 0; q0 < quads; q0 += 128) {
            f32x4 x[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
            for (int s0 = 0; s0 < a.splits; s0 += 8) {
                if (s0 != 0 || q0 != 0) load(s0, q0);
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const float f = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(pf), min(s0 + u, 63)));
                    if (s0 + u < a.splits) {
                        x[0] += y[u][0] * f;
                        x[1] += y[u][1] * f;
                    }
                }
            }
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const int quad = q0 + 64 * e + lane;
                if (quad >= quads) continue;
                uint32_t pw[3][2];
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    float r[2] = {x[e][2 * j] * inv, x[e][2 * j + 1] * inv};
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        const uint32_t c0 = float_to_bits<BF16>(r[0]), c1 = float_to_bits<BF16>(r[1]);
                        pw[q][j] = c0 | (c1 << 16);
                        r[0] = fabsf(r[0]) < INFINITY ? r[0] - bits_to_float(c0, BF16) : 0.0f;  // (an infinity or NaN is its first part)
                        r[1] = fabsf(r[1]) < INFINITY ? r[1] - bits_to_float(c1, BF16) : 0.0f;
                    }
                }
#pragma unroll
                for (int q = 0; q < 3; ++q) *reinterpret_cast<u32x2*>(op + (4 * q + wave) * lo + 4 * quad) = u32x2{pw[q][0], pw[q][1]};
            }
        }
    } else {
        weights(0);
    }
    __syncthreads();
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    const uint16_t* xo = op + min(l16, 11) * lo + 8 * g;
    for (int s0 = 0; s0 < steps; s0 += FLIGHT) {
        if (s0) weights(s0);
#pragma unroll
        for (int i = 0; i < FLIGHT; ++i)
            if (s0 + i < steps) acc = mfma16<BF16>(*reinterpret_cast<const u32x4*>(xo + 32 * (s0 + i)), w[i], acc);
    }
    // a lane holds column l16 and part g of the four tokens; lane group g finishes token g
    float x = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float t = __shfl(acc[i], l16) + (__shfl(acc[i], l16 + 16) + __shfl(acc[i], l16 + 32));
        x = g == i ? t : x;
    }
    if (a.gate) x *= sigmoid_f(gt);
    if (g < nb && v < a.vdim) reinterpret_cast<uint16_t*>(a.y)[(size_t)(b0 + g) * a.ldy + vc] = (uint16_t)float_to_bits<BF16>(x);
}

// sizes the matrix-core form of the single-token attention covers
inline bool step_on_matrix_cores(const int rank, const int ldq, const int dtype) {
    return (dtype == TEAL_BF16 || dtype == TEAL_F16) && rank <= 512 && ldq <= 32 * kStepKSteps;
}

template <bool TIED>
int launch_step(const StepAttentionArgs& a, const int batch, const size_t queries, const int dtype, hipStream_t st) {
    const int rt = a.rank <= 64 ? 4 : (a.rank <= 128 ? 8 : (a.rank <= 256 ? 16 : 32));
    const size_t lds = std::max(queries, (size_t)32 * step_tile_row(a.ldq, rt) * 2);  // (<= 41472 bytes)
    const dim3 grid(a.splits, a.heads / a.group * ((a.group + 15) / 16), batch), block(256);
#define TEAL_LD(BF, RT)                                                                                                \
    do {                                                                                                               \
        if (a.softcap > 0.0f) hipLaunchKernelGGL((step_attention_kernel<BF, RT, TIED, true>), grid, block, lds, st, a); \
        else hipLaunchKernelGGL((step_attention_kernel<BF, RT, TIED, false>), grid, block, lds, st, a);                \
    } while (0)
#define TEAL_LD_R(BF) do { if (rt == 4) TEAL_LD(BF, 4); else if (rt == 8) TEAL_LD(BF, 8); else if (rt == 16) TEAL_LD(BF, 16); else TEAL_LD(BF, 32); } while (0)
    if (dtype == TEAL_BF16) TEAL_LD_R(true);
    else TEAL_LD_R(false);
#undef TEAL_LD_R
#undef TEAL_LD
    return launched();
}

}  // namespace teal

using namespace teal;

extern "C" {

int teal_latent_prompt_rows(void* proj, int ldp, int kv0, int n_tokens, const int32_t* pos, const int32_t* row, const float* inv_freq, const void* norm_w,
                            float eps, int heads, int dim, int rot, int rank, void* cache, int ldc, int dtype, void* stream) {
    if (!proj || !pos || n_tokens <= 0 || heads <= 0 || dim < 0 || rot < 0 || dim + rot <= 0 || (rot > 0 && !inv_freq)) return TEAL_ERR_ARG;
    if (kv0 >= 0 && (!row || !norm_w || !cache || rank <= 0)) return TEAL_ERR_ARG;
    if ((rot & 1) || ldp < heads * (dim + rot) || (kv0 >= 0 && (kv0 < heads * (dim + rot) || ldp < kv0 + rank + rot || ldc < rank + rot))) return TEAL_ERR_SHAPE;
    const LatentRowArgs a = {proj, pos, row, inv_freq, norm_w, cache, ldp, kv0, heads, dim, rot, rank, ldc, eps};
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    return with_dtype(dtype, [&](auto dt) {
        hipLaunchKernelGGL((latent_prompt_rows_kernel<decltype(dt)::value>), dim3(n_tokens), dim3(256), 0, st, a);
        return launched();
    });
}

int teal_latent_gather(const void* cache, int ldc, const int32_t* row, int n_rows, int rank, int rot, void* c, void* kr, int dtype, void* stream) {
    if (!cache || !row || !c || (rot > 0 && !kr) || n_rows <= 0 || rank <= 0 || rot < 0) return TEAL_ERR_ARG;
    if (ldc < rank + rot) return TEAL_ERR_SHAPE;
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    return with_dtype(dtype, [&](auto dt) {
        using S = typename Num<decltype(dt)::value>::S;
        hipLaunchKernelGGL((latent_gather_kernel<decltype(dt)::value>), dim3(n_rows), dim3(64), 0, st, reinterpret_cast<const S*>(cache), ldc, row, rank, rot,
                           reinterpret_cast<S*>(c), reinterpret_cast<S*>(kr));
        return launched();
    });
}

int teal_layer_prompt_tile(int dim, int rot, int vdim, int n_queries, int dtype) {
    if (dtype == TEAL_F32 || dim + rot > 256 || vdim > 256) return 1;  // the scalar kernel: one query per workgroup
    return n_queries > 64 && vdim <= 128 ? 128 : 64;
}

int teal_layer_prompt_attention(const void* q, int ldq, const void* k, const void* kr, const void* vt, int n_keys, const void* sink, const void* gate,
                                int ldg, void* out, int ldo, const int32_t* seqs, const int32_t* tiles, int n_tiles, int tile, int heads, int group, int dim,
                                int rot, int vdim, int window, float scale, float softcap, int dtype, void* stream) {
    if (!q || !k || (rot > 0 && !kr) || !vt || !out || !seqs || !tiles || n_tiles <= 0 || heads <= 0 || dim < 0 || rot < 0 || vdim <= 0 || window <= 0) return TEAL_ERR_ARG;
    if (group <= 0 || heads % group) return TEAL_ERR_SHAPE;
    if (dim + rot <= 0 || dim + rot > 8192 || heads > 65535 || ldq < heads * (dim + rot) || ldo < heads * vdim || (gate && ldg < heads * vdim) || n_keys <= 0 || (n_keys & 7))
        return TEAL_ERR_SHAPE;
    if (tile != 1 && (dim + rot > 256 || vdim > 256 || (tile != 64 && tile != 128) || (tile == 128 && vdim > 128))) return TEAL_ERR_SHAPE;
    if (tile != 1 && (!aligned16(q) || !aligned16(k) || !aligned16(kr) || !aligned16(vt) || (reinterpret_cast<uintptr_t>(gate) & 7u) || (reinterpret_cast<uintptr_t>(out) & 7u)))
        return TEAL_ERR_ALIGN;
    if (tile != 1 && dtype == TEAL_F32) return TEAL_ERR_DTYPE;
    const PromptAttentionArgs a = {q, k, kr, vt, sink, gate, out, reinterpret_cast<const SeqSpan*>(seqs), tiles, ldq, gate ? ldg : 0, ldo, heads, group, dim, rot, vdim, n_keys, window, scale, softcap};
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (tile == 1)
        return with_dtype(dtype, [&](auto dt) {
            hipLaunchKernelGGL((prompt_attention_scalar_kernel<decltype(dt)::value>), dim3(n_tiles, heads), dim3(256), (size_t)(dim + rot + 512) * sizeof(float), st, a);
            return launched();
        });
    if (softcap > 0.0f) return launch_prompt_capped(a, tile, n_tiles, dtype, st);
    if (dtype == TEAL_BF16) return tile == 128 ? launch_prompt<true, 512, kCapNone>(a, n_tiles, st) : launch_prompt<true, 256, kCapNone>(a, n_tiles, st);
    if (dtype == TEAL_F16) return tile == 128 ? launch_prompt<false, 512, kCapNone>(a, n_tiles, st) : launch_prompt<false, 256, kCapNone>(a, n_tiles, st);
    return TEAL_ERR_DTYPE;
}

int teal_latent_step_query(const void* proj, int ldp, int kv0, int batch, const int32_t* pos, const int32_t* slot, const int32_t* table, int max_pages, int page_shift,
                           const float* inv_freq, const void* norm_w, float eps, const void* uk, int heads, int dim, int rot, int rank, void* cache, int ldc, void* qcat,
                           int ldq, int dtype, void* stream) {
    if (!proj || !pos || !slot || !table || !uk || !qcat || batch <= 0 || heads <= 0 || dim <= 0 || rot < 0 || rank <= 0 || max_pages <= 0 || (rot > 0 && !inv_freq)) return TEAL_ERR_ARG;
    if (kv0 >= 0 && (!norm_w || !cache)) return TEAL_ERR_ARG;
    if ((rot & 1) || dim > 8192 || batch > 65535 || page_shift < 5 || page_shift > 20 || (ldq & 31) || ldq < rank + rot || ldp < heads * (dim + rot) ||
        (kv0 >= 0 && (kv0 < heads * (dim + rot) || ldp < kv0 + rank + rot || ldc < rank + rot)))
        return TEAL_ERR_SHAPE;
    if (!aligned16(uk) || !aligned16(qcat)) return TEAL_ERR_ALIGN;
    const int chunks = (rank + 127) / 128;
    const LatentStepArgs a = {{const_cast<void*>(proj), pos, nullptr, inv_freq, norm_w, cache, ldp, kv0, heads, dim, rot, rank, ldc, eps}, slot, table, uk, qcat, max_pages, page_shift, chunks, ldq};
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    return with_dtype(dtype, [&](auto dt) {
        constexpr int DT = decltype(dt)::value;
        if constexpr (DT != TEAL_F32) {
            // (four tokens of 32 heads: 4.3 us against 3.8; six: 3.8 / 4.2; eight of 16 heads 3.9 / 6.5, six: the same)
            if (batch > 4 && batch * heads >= 128 && !(dim & 31) && !(rank & 15) && !(rot & 7) && !(ldp & 7) && rank <= 8192 && aligned16(proj)) {
                LatentStepArgs m = a;
                m.chunks = (rank + 255) / 256;
                hipLaunchKernelGGL((latent_step_query_rows_kernel<DT == TEAL_BF16>), dim3(heads * m.chunks + (kv0 >= 0 ? 16 : 0), (batch + 15) / 16), dim3(256), 0, st, m, batch);
                return launched();
            }
        }
        const int nx = heads * chunks + (kv0 >= 0 ? 1 : 0);
        // (from eight tokens on a workgroup reads its weights once for four of them)
        if (batch >= 8 && dim <= 2048) hipLaunchKernelGGL((latent_step_query_kernel<DT, 4>), dim3(nx, (batch + 3) / 4), dim3(256), (size_t)4 * dim * sizeof(float), st, a, batch);
        else hipLaunchKernelGGL((latent_step_query_kernel<DT, 1>), dim3(nx, batch), dim3(256), (size_t)dim * sizeof(float), st, a, batch);
        return launched();
    });
}

int teal_layer_step_attention(const void* qcat, int ldq, const void* cache, int ldc, const int32_t* pos, const int32_t* slot, const int32_t* table, int max_pages,
                              int page_shift, int batch, int heads, int group, int rank, int rot, int window, float scale, float softcap, int splits, float* part,
                              size_t part_bytes, int dtype, void* stream) {
    if (!qcat || !cache || !pos || !slot || !table || !part || batch <= 0 || heads <= 0 || rank <= 0 || rot < 0 || window <= 0 || max_pages <= 0) return TEAL_ERR_ARG;
    if (group <= 0 || heads % group || ldc < heads / group * ldq) return TEAL_ERR_SHAPE;
    if (splits < 1 || splits > kMaxStepSplits || batch > 65535 || heads > 65535 || page_shift < 5 || page_shift > 20 || (ldq & 31) || ldq < rank + rot || (ldc & 31) || rank + rot > 6144)
        return TEAL_ERR_SHAPE;
    if (!aligned16(qcat) || !aligned16(cache)) return TEAL_ERR_ALIGN;
    if (!aligned16(part)) return TEAL_ERR_ALIGN;
    if (part_bytes < (size_t)batch * heads * splits * part_stride(rank) * sizeof(float)) return TEAL_ERR_WORKSPACE;
    const StepAttentionArgs a = {qcat, cache, pos, slot, table, part, max_pages, page_shift, ldq, ldc, heads, group, rank, rot, window, splits, scale, softcap, nullptr, nullptr, 0, 0};
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    if (step_on_matrix_cores(rank, ldq, dtype)) return launch_step<false>(a, batch, 0, dtype, st);
    return with_dtype(dtype, [&](auto dt) {
        hipLaunchKernelGGL((step_attention_scalar_kernel<decltype(dt)::value>), dim3(splits, heads, batch), dim3(256), (size_t)(2 * rank + rot) * sizeof(float), st, a);
        return launched();
    });
}

int teal_grouped_step_attention(const void* proj, int ldp, int k0, int batch, const int32_t* pos, const int32_t* slot, const int32_t* table, int max_pages, int page_shift,
                                const float* inv_freq, int heads, int kv_heads, int dim, int rot, void* cache, int ldk, int window, float scale, float softcap, int splits,
                                void* qcat, float* part, size_t part_bytes, int dtype, void* stream) {
    if (!proj || !pos || !slot || !table || !cache || !part || batch <= 0 || heads <= 0 || kv_heads <= 0 || dim <= 0 || rot < 0 || max_pages <= 0 || window <= 0 ||
        (rot > 0 && !inv_freq))
        return TEAL_ERR_ARG;
    if ((rot & 1) || rot > dim || heads % kv_heads || k0 < heads * dim || ldp < k0 + kv_heads * dim || (ldk & 31) || ldk < dim + rot) return TEAL_ERR_SHAPE;
    const size_t lds = (size_t)std::min(16, heads / kv_heads) * 2 * ldk * 2;
    // (the static tiles of the largest kernel and the query rows share the 64 KB of a workgroup)
    if (!step_on_matrix_cores(dim, ldk, dtype) || lds > 16 * 1024) {
        if (!qcat) return TEAL_ERR_ARG;
        const int rc = teal_grouped_step_query(proj, ldp, k0, batch, pos, slot, table, max_pages, page_shift, inv_freq, heads, kv_heads, dim, rot, cache, ldk, qcat, ldk, dtype,
                                               stream);
        return rc != TEAL_OK ? rc : teal_layer_step_attention(qcat, ldk, cache, kv_heads * ldk, pos, slot, table, max_pages, page_shift, batch, heads, heads / kv_heads, dim, rot,
                                                              window, scale, softcap, splits, part, part_bytes, dtype, stream);
    }
    if (splits < 1 || splits > kMaxStepSplits || batch > 65535 || heads > 65535 || page_shift < 5 || page_shift > 20) return TEAL_ERR_SHAPE;
    if (!aligned16(cache) || !aligned16(part)) return TEAL_ERR_ALIGN;
    if (part_bytes < (size_t)batch * heads * splits * part_stride(dim) * sizeof(float)) return TEAL_ERR_WORKSPACE;
    const StepAttentionArgs a = {nullptr, cache, pos, slot, table, part, max_pages, page_shift, ldk, kv_heads * ldk, heads, heads / kv_heads, dim, rot, window, splits, scale,
                                 softcap, proj, inv_freq, ldp, k0};
    return launch_step<true>(a, batch, lds, dtype, reinterpret_cast<hipStream_t>(stream));
}

int teal_latent_step_merge(const float* part, int splits, const void* uv, const void* sink, const void* gate, int ldg, void* y, int ldy, int batch, int heads, int rank,
                           int vdim, int dtype, void* stream) {
    if (!part || !uv || !y || batch <= 0 || heads <= 0 || rank <= 0 || vdim <= 0 || splits < 1) return TEAL_ERR_ARG;
    if (splits > kMaxStepSplits || rank > 8192 || batch > 65535 || heads > 65535 || ldy < heads * vdim || (gate && ldg < heads * vdim)) return TEAL_ERR_SHAPE;
    if (!aligned16(uv) || !aligned16(part)) return TEAL_ERR_ALIGN;
    const LatentMergeArgs a = {part, uv, sink, gate, y, heads, rank, vdim, splits, ldg, ldy};
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    return with_dtype(dtype, [&](auto dt) {
        constexpr int DT = decltype(dt)::value;
        if constexpr (DT != TEAL_F32) {
            // (four tokens of 32 heads: 7.4 us against 8.7, three: the same; eight of 16 heads 7.4 / 16, six: 7.3 / 6.9)
            if (batch >= 4 && batch * heads >= 128 && !(rank & 31) && rank <= 2048 && vdim <= 65536) {
                hipLaunchKernelGGL((latent_merge_rows_kernel<DT == TEAL_BF16>), dim3((vdim + 63) / 64, heads, (batch + 3) / 4), dim3(256), (size_t)12 * (rank + 8) * 2, st, a, batch);
                return launched();
            }
        }
        const int nx = (vdim + 31) / 32;
        if (batch >= 8 && rank <= 2048) hipLaunchKernelGGL((latent_decode_merge_kernel<DT, 4>), dim3(nx, heads, (batch + 3) / 4), dim3(256), (size_t)(4 * ((rank + 7) & ~7) + 1024) * sizeof(float), st, a, batch);
        else hipLaunchKernelGGL((latent_decode_merge_kernel<DT, 1>), dim3(nx, heads, batch), dim3(256), (size_t)(((rank + 7) & ~7) + 1024) * sizeof(float), st, a, batch);
        return launched();
    });
}

}  // extern "C"
