/*
 * teal_hip.h — C ABI of libteal_hip.so, the MI355X (gfx950) implementation of TEAL's
 * activation-sparsity decode hot path.
 *
 * Every entry point replaces one piece of the reference's Triton path; citations are
 * into the reference tree (FasterDecoding/TEAL @ 2024-10-22):
 *
 *   teal_sparse_gemv       <- kernels/sparse_gemv.py:87-142  splitk_sparse_gemv()  + :50-83 kernel
 *                             (+ the init_to_zero("Y") pre-hook launch, :8-12, which disappears)
 *   teal_sparse_qkv_gemv   <- kernels/sparse_gemv.py:196-237 qkv_gemv()            + :152-194 kernel
 *   teal_compact           <- kernels/sparse_gemv.py:75      idx = tl.abs(x0) > threshold
 *                             (exposed standalone so index sets can be tested bit-exactly)
 *   teal_dense_gemv        <- kernels/sparse_gemv.py:301-307 DenseGEMV / torch.matmul(x, W.T) at S == 1
 *   teal_sparse_gateup_silu <- gpt-fast/model.py:258-259       silu(gemv1(x, w1)) * gemv1(x, w3)
 *   teal_fused_gemv        <- gpt-fast/model.py:158-161,289-291 residual adds + RMSNorm, :258-259 silu * up,
 *                             folded into the GEMV launch as producers
 *   teal_decode_attention* <- gpt-fast/model.py:170-186       RoPE, kv_cache.update, SDPA at S == 1
 *                             (TEAL_OUT_QKV_ROPE + teal_decode_attention_split_roped: RoPE and the cache append in the wqkv
 *                             projection's epilogue, :170-178, SDPA in the attention launch)
 *   teal_sample_topk       <- gpt-fast/generate.py:49-66      logits_to_probs + multinomial_sample_one
 *   teal_sparse_qkv_gemv_i8 <- gpt-fast/quantize.py:339-357   WeightOnlyInt8Linear.forward on the masked x
 *   teal_sparse_qkv_gemv_i4 <- gpt-fast/quantize.py:58-162,483-526 group-quantised int4 linear on the masked x
 *   teal_cmp_flag_gemv     <- scripts/benchmark_gemv.py:32-107,170-172 the Deja Vu comparator of the kernel benchmark
 *   teal_prefill_*         <- kernels/sparse_gemv.py:271,298 (dense matmul when S > 1) + gpt-fast/model.py:107-121,158-186,258-259:
 *                             the prompt pass of a short prompt, counted by the reference's tokens/sec (generate.py:458,487-496)
 *
 * Conventions
 *   - extern "C", plain pointers and sizes, no C++/torch types, no exceptions across the boundary.
 *   - All pointers are DEVICE pointers owned by the caller (PyTorch); the library borrows them for
 *     the duration of the stream-ordered launch and never allocates.  Library state: the properties of each device,
 *     cached the first time it is used (teal_init(); immutable), and a host-side registry of the workspaces prepared by
 *     teal_workspace_init() (which device memory holds a valid header; mutex-protected).  Nothing else: no entry point
 *     of libteal_hip.so changes how a later call behaves, and what a call did is reported through its own arguments
 *     (teal_gemv_out_t.desc).  The tuning / phase-stamp switches of the last section exist only in the DIAGNOSTICS
 *     build of the same sources, libteal_hip_diag.so (-DTEAL_DIAGNOSTICS), which the product path never loads.
 *     No device memory belongs to the library: the arrival counters of the single-launch split-K GEMVs and the scratch of the
 *     multi-workgroup sampler live in the header of the CALLER's workspace, so two streams, two captured graphs or two
 *     devices can only collide if the caller hands them the same workspace.
 *   - `stream` is a hipStream_t passed as void* (0 = the null stream).  Every call is
 *     asynchronous, allocation-free and hipGraph-capture safe.
 *   - dtype: 0 = fp16, 1 = bf16 (x, weights and y share it; int8 weights carry scales in that dtype).
 *   - Weight layout: the reference's "column major" weight[N, Z] with strides (1, N), i.e. the
 *     memory image is W^T row-major [Z][N]: element (m, n) at wT[m * N + n]
 *     (kernels/sparse_gemv.py:68,106).  N % 8 == 0 (16-byte rows), 1 <= Z <= 65536.
 *   - Keep rule: row m is kept iff float32(|x[m]|) > float32(tau)  (strict; kernels/sparse_gemv.py:75).
 *     In the GEMV entry points a NaN x[m] additionally propagates NaN into every output column of its
 *     threshold group, as the reference's `0 * NaN` on masked rows does.
 *   - Arithmetic: fp32 multiply-accumulate over the kept rows, ONE rounding to dtype at the end
 *     (the reference rounds through fp16 atomics, kernels/sparse_gemv.py:83); no atomics, results are
 *     bit-reproducible run to run.
 *   - Return value: 0 on success, negative TEAL_ERR_* otherwise (teal_strerror()).
 */
#ifndef TEAL_HIP_H
#define TEAL_HIP_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define TEAL_OK 0
#define TEAL_ERR_ARG (-1)       /* null pointer / non-positive size */
#define TEAL_ERR_DTYPE (-2)     /* dtype not 0 (fp16) / 1 (bf16) */
#define TEAL_ERR_SHAPE (-3)     /* N % 8 != 0, Z > 65536, bad N_q / N_kv */
#define TEAL_ERR_ALIGN (-4)     /* pointer not 16-byte aligned */
#define TEAL_ERR_WORKSPACE (-5) /* workspace too small (teal_workspace_bytes) */
#define TEAL_ERR_LAUNCH (-6)    /* hipGetLastError() after the launch */
#define TEAL_ERR_NO_DEVICE (-7) /* no HIP device / teal_init failed */
#define TEAL_ERR_CONFIG (-8)    /* invalid tuning override */

#define TEAL_F16 0
#define TEAL_BF16 1
#define TEAL_F32 2 /* the layered designs' entry points only (teal_layer_*, teal_gated_act, teal_logit_softcap, teal_latent_*,
                    * teal_grouped_*, teal_wkv_*) */

int teal_version(void);
const char* teal_strerror(int code);

/* Cache the immutable properties of the CURRENT device (CU count, per-kernel attributes).  Call once per device
 * before any launch that may happen during stream capture (every entry point does it lazily otherwise).  Returns the
 * CU count (> 0) or a negative error. */
int teal_init(void);

/* Bytes of workspace a GEMV with N output columns may need: the library's header (arrival counters, sampler scratch)
 * plus an upper bound of the fp32 split-K slabs over all launch geometries (the deepest split x two N-column
 * segments).  Does not depend on Z — accepted for symmetry with the GEMV entry points.  The caller allocates once and
 * reuses; distinct streams need distinct workspaces. */
size_t teal_workspace_bytes(int Z, int N);

/* Prepare a workspace: zero its header (asynchronously on `stream`) and remember the pointer.  Once per allocation,
 * before the first launch that uses it and not under stream capture.  A prepared workspace lets a split-K GEMV with a
 * rounded output run as ONE launch (per-tile arrival tickets; the last slice to arrive sums the partials in slice
 * order) and a large-vocabulary sampler as several workgroups; every launch re-arms what it used, so a graph that was
 * captured with the workspace can be replayed indefinitely.  An unprepared workspace (plain memory of
 * teal_workspace_bytes) is still valid everywhere: 16-bit weights give the SAME bits from GEMV + ordered reduce launch (the
 * same slices summed in the same order) and the sampler the same tokens from a single workgroup; int8 / int4 weights pick
 * their split-K factor by whether tickets are available, so there the two ways agree to the tolerance of the fp32
 * summation order (one ulp of the 16-bit output), not bit for bit.  If a launch is aborted (device reset), prepare again.  teal_workspace_release() forgets the
 * pointer; call it before freeing the memory. */
int teal_workspace_init(void* ws, size_t ws_bytes, void* stream);
int teal_workspace_release(void* ws);

/* idx_out[0..count) = ascending m with float32(|x[m]|) > float32(tau); *count_out = count.
 * idx_out must hold Z int32.  (kernels/sparse_gemv.py:75) */
int teal_compact(const void* x, float tau, int Z, int dtype, int32_t* idx_out, int32_t* count_out,
                 void* stream);

/* y[n] = sum_{m kept} wT[m*N + n] * x[m]            (kernels/sparse_gemv.py:87-142) */
int teal_sparse_gemv(const void* x, const void* wT, void* y, float tau, int Z, int N, int dtype,
                     void* ws, size_t ws_bytes, void* stream);

/* Same on the fused wqkv weight with a threshold per column range:
 * columns [0,N_q) tau_q, [N_q,N_q+N_kv) tau_k, [N_q+N_kv,N) tau_v   (kernels/sparse_gemv.py:196-237;
 * N_q = N - 2*kv_size, N_kv = kv_size there).  N_q and N_kv must be multiples of 8. */
int teal_sparse_qkv_gemv(const void* x, const void* wT, void* y, float tau_q, float tau_k,
                         float tau_v, int Z, int N, int N_q, int N_kv, int dtype, void* ws,
                         size_t ws_bytes, void* stream);

/* Same with an explicit row stride `ld >= N` (elements, multiple of 8) of the W^T image, i.e. weight[N, Z]
 * with strides (1, ld).  A stride that is NOT a multiple of 1024 bytes (ld = N + 64) makes consecutive
 * rows start in different 128-byte DRAM-channel residues, so a workgroup's column tile rotates over all
 * channels instead of hammering one. */
int teal_sparse_qkv_gemv_ld(const void* x, const void* wT, int ld, void* y, float tau_q, float tau_k,
                            float tau_v, int Z, int N, int N_q, int N_kv, int dtype, void* ws,
                            size_t ws_bytes, void* stream);

/* int8 weight-only variant of teal_sparse_qkv_gemv_ld (the reference ships int8 only for its
 * dense path, gpt-fast/quantize.py:339-357, and lists quantised TEAL as missing, README.md:110).  wqT = int8 image of
 * W^T, row-major [Z][ld] bytes (ld % 8 == 0, ld >= N); scale[N] in the activation dtype.  N_kv = 0, N_q = N: one
 * threshold (tau_q). */
int teal_sparse_qkv_gemv_i8(const void* x, const void* wqT, const void* scale, void* y, float tau_q, float tau_k,
                            float tau_v, int Z, int N, int N_q, int N_kv, int ld, int dtype, void* ws, size_t ws_bytes,
                            void* stream);

/* y = x @ W^T with every row kept (prefill-free decode of un-sparsified layers, e.g. lm_head).
 * (kernels/sparse_gemv.py:301-307) */
int teal_dense_gemv(const void* x, const void* wT, void* y, int Z, int N, int dtype, void* ws,
                    size_t ws_bytes, void* stream);

/* int4 group-quantised weight-only variant (the reference ships int4-g32/64/128/256 for its dense
 * path only: gpt-fast/quantize.py:58-162 group q-params / quantise / dequantise, :483-526 WeightOnlyInt4Linear over a
 * CUDA-only packed layout).  w[n][m] = (q - 8) * scale[m / G][n] + zero[m / G][n], q in 0..15.
 *   wq               nibble image of W^T by ROW PAIRS: [Z / 2][ldb] BYTES (ldb >= N, ldb % 8 == 0, 8-byte aligned; for speed
 *                    ldb % 128 == 0 and a 128-byte aligned base, so that a tile's 128-byte segment is ONE memory line); the
 *                    32-bit word g of pair-row p holds columns 4g .. 4g+3 of row 2p in its low half (nibble j = column
 *                    4g + j) and of row 2p + 1 in its high half — two rows of a column unpack into one half2 for a packed
 *                    dot product; a pair is fetched when either of its rows is kept
 *   scales_and_zeros bf16 [Z / G][N][2] = {scale, zero}, exactly the reference's tensor (quantize.py:79-93)
 * N, N_q, N_kv multiples of 128; Z a multiple of G; x / y fp16 or bf16 (dtype).  N_kv = 0, N_q = N: one threshold.
 * One launch (split-K over 32-row units folded in by arrival tickets); fp32 accumulation, scale / zero applied once per
 * (unit, column), one rounding. */
int teal_sparse_qkv_gemv_i4(const void* x, const void* wq, const void* scales_and_zeros, void* y, float tau_q, float tau_k,
                            float tau_v, int Z, int N, int N_q, int N_kv, int ldb, int groupsize, int dtype, void* ws,
                            size_t ws_bytes, void* stream);

/* ---- fusions around the path ------------------------------------------ */

/* h[n] = silu(gate[n]) * up[n] with gate = sparse_gemv(x, w1T, tau_gate), up = sparse_gemv(x, w3T,
 * tau_up), both [Z][N]; gate/up are rounded to dtype before the activation and the product, as the
 * unfused reference sequence does (gpt-fast/model.py:258-259).  One launch, one shared read of x. */
int teal_sparse_gateup_silu(const void* x, const void* w1T, const void* w3T, void* h, float tau_gate,
                            float tau_up, int Z, int N, int dtype, void* ws, size_t ws_bytes,
                            void* stream);

/* ---- fused decode step: producers/consumers folded into the GEMV launch - */

#define TEAL_IN_PLAIN 0      /* x given as is */
#define TEAL_IN_RESID_NORM 1 /* x = RMSNorm(resid + round(sum slabs)) * w   (model.py:158-161, 289-291) */
#define TEAL_IN_SILU_MUL 2   /* x = silu(gate) * up, gate|up contiguous [2Z] (model.py:258-259) */
#define TEAL_IN_MASKED 3     /* x given together with its keep masks (one uint64 per 64 elements, bit i =
                              * element 64*c+i kept) as emitted by the producing launch: the consumer skips
                              * the compare/ballot phase.  The masks must be those of tau[0]. */
#define TEAL_IN_ATTN_MERGE 4 /* x = attention output merged from the split-KV partials per head written by
                              * teal_decode_attention_split(y = NULL, nsplit = 4 or 8): x points at the fp32
                              * partials [Z/head_dim][nsplit][head_dim + 2]; att_head_dim = head_dim,
                              * att_nsplit = nsplit (0 means 4); Z <= 16384 (nsplit 4) / 8192 (nsplit 8) */
#define TEAL_IN_RESID32_NORM 5 /* the layered designs' residual, held in fp32: x = resid + y * (1 / rms(y)) * post, y = sum slabs + bias
                              * (no slabs: x = resid), then RMSNorm(x) * pre.  resid_in fp32 [Z] (with row_index: the 16-bit table
                              * [rows][Z]), norm_weight = three 16-bit vectors [3][Z] = pre | post | bias, resid_out fp32 [Z]; slabs
                              * interleaved.  Z % 64 == 0, Z <= 8192, segments whole 64-column tiles of 16-bit weights; other shapes
                              * return TEAL_ERR_CONFIG without launching.  Out modes ROUNDED, SLABS, SLAB_SUM */
#define TEAL_OUT_ROUNDED 0   /* y rounded to dtype (runs the ordered slab reduce when split-K is used) */
#define TEAL_OUT_SLABS 1     /* leave the fp32 split-K slabs for the next launch's RESID_NORM producer */
#define TEAL_OUT_QKV_ROPE 3  /* nseg == 3 = q | k | v of ONE fused wqkv image, RESID_NORM input: when the launch needs no
                              * split-K (and the lean kernel takes it: *nslabs_out = 0), its epilogue applies RoPE to q and
                              * to the new k row and appends k, v to the caches (gpt-fast/model.py:170-178): y[0] = rotated
                              * q [ncols[0]], rounded exactly as teal_decode_attention* would have; follow it with
                              * teal_decode_attention_split_roped.  Otherwise (*nslabs_out >= 1) the launch behaved as
                              * TEAL_OUT_SLABS (slabs required) and teal_decode_attention_split_slabs finishes the job */
#define TEAL_OUT_SLAB_SUM 4  /* nseg == 1: `slabs` (plain memory, fp32 [ncols]) receives the UNROUNDED sum over the row slices,
                              * added in slice order by the last slice of each tile to arrive (arrival tickets: `ws` must be a
                              * prepared workspace when the launch uses split-K) — bit-identical to summing the TEAL_OUT_SLABS
                              * slabs in slice order.  *nslabs_out = 1; the consumer is a RESID_NORM producer with nslabs = 1,
                              * slabs_interleaved = 0.  Tensor parallelism: the [ncols] fp32 vector is what the ranks all-reduce
                              * (gpt-fast/tp.py:120-121,139-140) instead of [ncols][4..8] slabs.  16-bit and int8 weights; shapes
                              * outside the lean kernel return TEAL_ERR_CONFIG without launching */
#define TEAL_OUT_PAIR_SILU 2 /* nseg == 2 (gate, up of equal shape): every workgroup streams the same column tile
                              * of both matrices and stores h = silu(gate) * up to y[0] (model.py:258-259); optional
                              * mask_out[ncols/64] = keep masks of h against mask_tau for a TEAL_IN_MASKED consumer */

typedef struct teal_gemv_in {
    int mode;                 /* TEAL_IN_* */
    const void* x;            /* PLAIN: [Z];  SILU_MUL: gate[Z] followed by up[Z] */
    const void* resid_in;     /* RESID_NORM: residual stream [Z] (or a [rows][Z] table with row_index) */
    const int32_t* row_index; /* RESID_NORM, optional: device int32; row = row_index[0] (embedding lookup) */
    const float* slabs;       /* RESID_NORM, optional: fp32 [nslabs][Z] partial sums folded into the residual */
    int nslabs;
    const void* norm_weight;  /* RESID_NORM: RMSNorm weight [Z] */
    float eps;
    void* resid_out;          /* RESID_NORM, optional: updated residual [Z]; must not alias resid_in */
    const void* masks;        /* MASKED: uint64 [ceil(Z/64)] keep masks of x */
    int att_head_dim;         /* ATTN_MERGE: head_dim */
    int att_nsplit;           /* ATTN_MERGE: partials per head, 4 or 8 (0 = 4) */
    int slabs_interleaved;    /* RESID_NORM: slabs are [Z][(nslabs+3)&~3] (as written by a producer with
                               * slabs_interleaved = 1) instead of planar [nslabs][Z]; nslabs <= 8 */
    int gate_activated;       /* SILU_MUL: the gate half already holds round(silu(gate)) — written by a launch with
                               * act_seg0 = 1 — so x = round(gate * up): the same roundings as the unfused sequence
                               * (model.py:258-259), the activation computed once per column instead of in every consumer
                               * workgroup's prologue.  16-bit and int8 weights (not the int4 kernel) */
    /* RESID32_NORM only (zero otherwise): */
    int no_post_norm;         /* 1: x = resid + y, the post vector is not used */
    float norm_offset;        /* added to the post and pre weights */
    /* token shift (teal_wkv_mix in the producer): column block s = min(column / mix_cols, mix_n - 1) of the output reads
     * h + (previous h - h) * mix_mu[s], h in fp32; the previous h comes from shift[slot][(pos - 1) & 1], this h goes to
     * shift[slot][pos & 1].  mix_cols % 64 == 0; mix_mu 16-bit [mix_n][Z]; shift fp32 [slots][2][Z] */
    const void* mix_mu;
    int mix_cols, mix_n;
    float* shift;
    const int32_t* shift_pos;  /* device int32 [1] */
    const int32_t* shift_slot; /* device int32 [1] */
} teal_gemv_in_t;

typedef struct teal_gemv_out {
    int nseg;            /* 1..3 column segments, each with its own threshold (q|k|v, gate|up, ...) */
    const void* w[3];    /* weight image of the segment: row-major [Z][ld] */
    int ld[3];           /* row stride (elements) */
    int col0[3];         /* first column of the segment inside a row */
    int ncols[3];        /* columns in the segment */
    float tau[3];        /* keep threshold of the segment */
    void* y[3];          /* ROUNDED: output of the segment [ncols] */
    int mode;            /* TEAL_OUT_* */
    float* slabs;        /* SLABS: destination, fp32 [nslabs][sum ncols]; plain memory, NOT a prepared workspace */
    size_t slabs_bytes;
    void* mask_out;      /* PAIR_SILU, optional: uint64 [ceil(ncols/64)] keep masks of h */
    float mask_tau;      /* PAIR_SILU: threshold of the consumer (the down projection) */
    int slabs_interleaved; /* SLABS: write slabs[col][slice] with row stride (nslabs+3)&~3 so that the consumer
                            * fetches every partial of an element with one 16-byte load */
    int weight_bits;       /* 0 or 16: fp16/bf16 weights (the activation dtype); 8: int8 weight-only quantisation
                            * (gpt-fast/quantize.py:339-357): w[i] = int8 image of W^T, row-major [Z][ld] BYTES, and
                            * scale[i] = per-output-column scales in the activation dtype (element 0 = column col0[i]);
                            * y = round(fp32(sum q*x) * fp32(scale)) — one rounding, where the reference's
                            * F.linear(x, w.to(dtype)) * scales rounds twice */
    const void* scale[3];  /* int8: see above.  int4 (weight_bits = 4, gpt-fast/quantize.py:58-162, 483-526): w[i] = packed image
                            * of W^T by row pairs, [Z / 2][ld BYTES] (see teal_sparse_qkv_gemv_i4); scale[i] = the
                            * reference's scales_and_zeros tensor of that image, bf16 [Z / groupsize][scale_ld[i]][2]; col0
                            * addresses both.  ncols multiples of 128; in modes PLAIN, RESID_NORM (interleaved slabs, <= 8),
                            * SILU_MUL, ATTN_MERGE; out modes ROUNDED and SLABS */
    int scale_ld[3];       /* int4 only: columns per group row of scale[i] (the image's N) */
    int groupsize;         /* int4 only: 32, 64, 128 or 256 rows per quantisation group; Z a multiple */
    /* TEAL_OUT_QKV_ROPE only (zero otherwise): */
    const void* rope;          /* (cos, sin) table [rope_max_seq][rope_head_dim / 2][2], activation dtype */
    const int32_t* rope_pos;   /* device int32: position of the token being decoded (clamped to the cache) */
    void* k_cache;             /* [ncols[1] / rope_head_dim][rope_max_seq][rope_head_dim] */
    void* v_cache;
    int rope_head_dim;         /* 64 or 128 */
    int rope_max_seq;
    int act_seg0;              /* TEAL_OUT_ROUNDED: y[0] = round(silu(round(sum))) for segment 0 (the gate projection of an
                                * unpaired gate | up launch, model.py:258); the other segments are stored as usual.  16-bit
                                * and int8 weights (not the int4 kernel) */
    char* desc;                /* optional HOST buffer: receives the kernel template instantiation and grid of the launch THIS
                                * call made, NUL-terminated (as rocprofv3 prints it; e.g. to name the kernel in a benchmark
                                * record) — per call, no library state */
    int desc_bytes;            /* capacity of desc (160 is enough) */
    /* TEAL_IN_RESID32_NORM launches only (zero otherwise), ROUNDED and SLAB_SUM outputs: */
    const void* bias;          /* 16-bit [sum ncols]: added to the complete sums; act_seg0 = 2 then applies gelu (tanh form) to
                                * segment 0, act_seg0 = 3 max(z, 0)^2 */
    float softcap;             /* > 0: the output is softcap * tanh(sum / softcap) */
} teal_gemv_out_t;

/* One launch: [fused producer] -> mask + compaction -> gathered GEMV over every segment.
 * *nslabs_out receives the split-K factor used (the number of slabs written in SLABS mode). */
int teal_fused_gemv(const teal_gemv_in_t* in, const teal_gemv_out_t* out, int Z, int dtype, void* ws,
                    size_t ws_bytes, int* nslabs_out, void* stream);

/* Single-token attention between gemv1 and gemv2 (gpt-fast/model.py:170-186): RoPE(q, k_new) with the
 * (cos, sin) table rope[max_pos][head_dim/2][2], KV-cache append at *pos, softmax(q K^T / sqrt(d)) V.
 * qkv = [q | k | v] as produced by the fused wqkv GEMV; caches are [n_kv_head][max_seq][head_dim];
 * y = [n_head * head_dim].  head_dim 64 or 128.  A position >= max_seq is clamped to the last cache slot (no
 * out-of-bounds write; the output of such a step is meaningless). */
int teal_decode_attention(const void* qkv, const void* rope, const int32_t* pos, void* k_cache, void* v_cache,
                          void* y, int n_head, int n_kv_head, int head_dim, int max_seq, int dtype, void* stream);

/* Same, also emitting the keep masks of y against mask_tau (uint64 [n_head*head_dim/64]) for a
 * TEAL_IN_MASKED wo projection. */
int teal_decode_attention_masked(const void* qkv, const void* rope, const int32_t* pos, void* k_cache, void* v_cache,
                                 void* y, void* mask_out, float mask_tau, int n_head, int n_kv_head, int head_dim,
                                 int max_seq, int dtype, void* stream);

/* Long-context form (flash-decoding): the cached positions of every head are split over `nsplit` workgroups
 * that write un-normalised partials {max, sum, o[head_dim]} (fp32, n_head*nsplit*(head_dim+2) floats), then
 * a merge launch rescales, sums, rounds once and emits the masks.  Use when max_seq is in the thousands:
 * one workgroup per head would leave most CUs idle while n_head of them stream the whole KV cache.
 * nsplit <= 64.  Grouped-query shapes (n_head / n_kv_head = 8 with max_seq >= 2048, = 4 with max_seq >= 4096) run as ONE workgroup per
 * (KV head, split) that serves all query heads of the group, so every K/V row is read once instead of once per query
 * head; choose nsplit so that n_kv_head * nsplit is about the CU count (32 for 8 KV heads).  Same partial format. */
int teal_decode_attention_split(const void* qkv, const void* rope, const int32_t* pos, void* k_cache, void* v_cache,
                                void* y, void* mask_out, float mask_tau, int n_head, int n_kv_head, int head_dim,
                                int max_seq, int nsplit, void* partials, size_t partials_bytes, int dtype, void* stream);
/* Same, with the qkv projection taken from the fp32 split-K slabs of a TEAL_OUT_SLABS launch (slabs_interleaved = 1,
 * layout [col][(nslabs + 3) & ~3], nslabs <= 8): the kernel sums each element's partials in slice order and rounds
 * once — exactly what the ordered reduce launch would have written — so a narrow (GQA) wqkv can be row-sliced over
 * all CUs without a reduce launch between projection and attention. */
int teal_decode_attention_split_slabs(const float* qkv_slabs, int qkv_nslabs, const void* rope, const int32_t* pos,
                                      void* k_cache, void* v_cache, void* y, void* mask_out, float mask_tau, int n_head,
                                      int n_kv_head, int head_dim, int max_seq, int nsplit, void* partials,
                                      size_t partials_bytes, int dtype, void* stream);
/* General form: exactly one of qkv (rounded projection) / qkv_slabs (+ qkv_nslabs) is given.  Same launches and results as
 * teal_decode_attention_split / _split_slabs.  `ws` / `ws_bytes` are accepted and unused (round 3 folded the merge launch into
 * the split launch through arrival counters in a prepared workspace: bit-identical y, measured no faster — equal at 4-8
 * splits, slower at 16-32 — and removed in round 5). */
int teal_decode_attention_split_ws(const void* qkv, const float* qkv_slabs, int qkv_nslabs, const void* rope,
                                   const int32_t* pos, void* k_cache, void* v_cache, void* y, void* mask_out,
                                   float mask_tau, int n_head, int n_kv_head, int head_dim, int max_seq, int nsplit,
                                   void* partials, size_t partials_bytes, int dtype, void* ws, size_t ws_bytes, void* stream);
/* After a TEAL_OUT_QKV_ROPE projection that reported *nslabs_out = 0: q = the rotated, rounded query [n_head * head_dim];
 * the token's k / v rows are already in the caches.  Always the per-query-head split kernel (no grouped-query form); same
 * partials, merge and results as teal_decode_attention_split_ws. */
int teal_decode_attention_split_roped(const void* q, const int32_t* pos, const void* k_cache, const void* v_cache, void* y,
                                      void* mask_out, float mask_tau, int n_head, int n_kv_head, int head_dim, int max_seq,
                                      int nsplit, void* partials, size_t partials_bytes, int dtype, void* ws, size_t ws_bytes,
                                      void* stream);
/* y == NULL: only the partials are written (no merge launch); with nsplit 4 or 8 a TEAL_IN_ATTN_MERGE wo
 * projection merges them in its own prologue (nsplit 4 or 8) — one launch less per layer, and 4 CUs per head pull the KV
 * cache instead of one (a single CU sustains ~50 GB/s, which bounds the one-workgroup-per-head kernel). */

/* Sampling step of the decode loop (gpt-fast/generate.py:49-66): logits / temperature, top-k filter
 * (ties at the pivot kept), softmax, exponential-race multinomial.  rng_state = device uint64[2]
 * {seed, draw counter}; the kernel bumps the counter so hipGraph replays draw fresh numbers.
 * top_k <= 0 or >= vocab disables the filter.  token_out = device int32[1] (may be the buffer the next
 * decode step reads its token from).  Optional in-graph loop-carried state, so that one graph replay
 * IS one decode step with no host-side glue: pos_inout[0] += 1; history[draw counter] = token.
 * teal_sample_topk_ws with a prepared workspace (teal_workspace_init): vocabularies of 8193..131072 entries (multiple
 * of 8) with an active filter run as one workgroup per 8192 logits: local top-k candidates -> workspace header -> the
 * last workgroup to arrive picks the token; same tokens as the single-workgroup kernels, which serve every other case
 * (no / unprepared workspace, other shapes). */
int teal_sample_topk(const void* logits, int vocab, int dtype, int top_k, float temperature, void* rng_state,
                     int32_t* token_out, int32_t* pos_inout, int32_t* history, int history_len, void* stream);
int teal_sample_topk_ws(const void* logits, int vocab, int dtype, int top_k, float temperature, void* rng_state,
                        int32_t* token_out, int32_t* pos_inout, int32_t* history, int history_len, void* ws,
                        size_t ws_bytes, void* stream);


/* ---- dense prompt pass for short prompts (T <= 16 tokens), teal_amd/csrc/teal_prefill.hip ----- */

/* The reference's prefill is dense (its ops run torch.matmul when the sequence is longer than one token,
 * kernels/sparse_gemv.py:271,298; the rest is the stock model, gpt-fast/model.py:107-121,158-186,258-259,289-291) and its
 * tokens/sec counts it (gpt-fast/generate.py:458,487-496).  These entry points make one layer of that pass seven launches over
 * the decode step's own weight images.  Every hand-over is TRANSPOSED, [feature][R] with R = 8 for T <= 8 and R = 16 for
 * 9 <= T <= 16 (every call of one pass takes the same T, hence the same R; "[..][8]" below reads "[..][R]"): the tokens of a
 * feature in one or two 16-byte words (16-bit activations: xt, ht, yt) or R / 4 of them (fp32 slabs [slice][feature][R]); token
 * slots >= T of the 16-bit vectors are written as zero, of the slabs left untouched (consumers ignore them).  1 <= T <= 16.
 * Floating-point results: fp32 sums, the rounding points of the module path's 16-bit tensors. */

/* What a GEMM launch builds its activations from (every workgroup builds the rows of its own slice, once, while staging them) */
#define TEAL_PREFILL_IN_XT 0        /* xt [Z][8] as given */
#define TEAL_PREFILL_IN_NORM 1      /* x = RMSNorm(h) * norm_w from the residual rows xt = ht [Z][8] and the per-workgroup sums of squares
                                     * sumsq [nwg][8] a teal_prefill_resid_norm call left in its scratch (nwg = Z / 256 rounded up) */
#define TEAL_PREFILL_IN_SILU_MUL 2  /* x = round(round(silu(round(gate))) * round(up)) from the slabs [gu_split][2 Z][8] of a gate | up launch */
typedef struct teal_prefill_in {
    int mode;
    const void* xt;
    const float* sumsq;
    int nwg;
    const void* norm_w;
    float eps;
    const float* gu_slabs;
    int gu_split;
} teal_prefill_in_t;

/* slabs[slice][n][s] = sum over the slice's rows m of W^T[m][n] * x[m][s]: w0T [Z][ld0] (n0 columns) and, optionally, w1T [Z][ld1]
 * (n1 columns, output columns n0 ..: gate | up in one launch).  Z, n0, n1 multiples of 256.  *split_out = slices written (<= 16;
 * the consumer sums them in slice order and rounds once); slabs must hold 16 * (n0 + n1) * R floats and must not be the buffer a
 * TEAL_PREFILL_IN_SILU_MUL launch reads. */
int teal_prefill_gemm(const teal_prefill_in_t* in, const void* w0T, int ld0, int n0, const void* w1T, int ld1, int n1, float* slabs,
                      size_t slabs_bytes, int Z, int T, int dtype, int* split_out, void* stream);
/* h = (embedding rows of tokens[0..T) | ht_in) + round(sum of `split` slabs) (split 0: nothing to add); x = RMSNorm(h) * norm_w.
 * Exactly one of tokens (+ emb [vocab][dim]) / ht_in is given; with neither xt_out nor x_last only the first of the two launches runs
 * (h and the sums of squares: a TEAL_PREFILL_IN_NORM GEMM normalises while it stages).  Outputs: ht_out [dim][8] (required; must not alias ht_in's
 * words of other columns — the same buffer is fine), xt_out [dim][8] and x_last [dim] (optional) = the normalised vector of
 * token T - 1 as a plain vector (input of the lm_head GEMV).  sumsq_scratch: (dim / 256 rounded up) * R floats of caller memory
 * (the per-workgroup sums of squares between the two launches this call makes).  dim <= 16384. */
int teal_prefill_resid_norm(const void* emb, const int32_t* tokens, int T, const void* ht_in, const float* slabs, int split,
                            const void* norm_w, float eps, int dim, void* ht_out, void* xt_out, void* x_last, float* sumsq_scratch,
                            int dtype, void* stream);
/* q | k | v from the slabs [split][(n_head + 2 n_kv_head) * head_dim][8] of the wqkv launch: RoPE(q, k) at positions 0 .. T-1,
 * cache rows 0 .. T-1 written, causal softmax(q K^T / sqrt(d)) V -> yt [n_head * head_dim][8].  head_dim 64 or 128. */
int teal_prefill_attention(const float* qkv_slabs, int split, const void* rope, void* k_cache, void* v_cache, void* yt, int T, int n_head,
                           int n_kv_head, int head_dim, int max_seq, int dtype, void* stream);

/* ---- Llama prompt pass of any length, teal_amd/csrc/teal_prompt.hip ----------------------------------------------------
 * 16-bit rows [token][feature]; the rounding points are the module path's 16-bit tensors.  Positions and token ids are device int32 or int64
 * arrays ([T]; the ..64 flags) and are kept inside their tables. */

/* h[t] = (emb[tokens[t]] | h[t]) + (y[t] | round(sum of n_slabs fp32 slabs [n_slabs][T][dim])); x[t] = RMSNorm(h[t]) * w.  emb / y / slabs optional; dim
 * % 8 == 0, <= 16384; zero: optional, n_zero <= 256 counters set to zero */
int teal_prompt_norm(const void* emb, int vocab, const void* tokens, int tokens64, void* h, const void* y, const float* slabs, int n_slabs, const void* w,
                     void* x, int T, int dim, float eps, unsigned* zero, int n_zero, int dtype, void* stream);
/* qkv [T][ldq] = q | k | v: q rotated in place, k rotated and v into the rows pos[t] of the caches [n_kv_head][max_seq][head_dim] */
int teal_prompt_rope(void* qkv, int ldq, const void* rope, const void* pos, int pos64, void* k_cache, void* v_cache, int T, int n_head, int n_kv_head,
                     int head_dim, int max_seq, int dtype, void* stream);
/* out[t] = softmax(scale * q[t] K^T) V over the cache rows 0 .. pos[t]; head_dim 64 or 128 */
int teal_prompt_attention(const void* q, int ldq, const void* k_cache, const void* v_cache, const void* pos, int pos64, void* out, int ldo, int T,
                          int n_head, int n_kv_head, int head_dim, int max_seq, float scale, int dtype, void* stream);
/* h[i] = round(silu(gate[i])) * up[i], i < n (n % 8 == 0) */
int teal_silu_mul(const void* gate, const void* up, void* h, size_t n, int dtype, void* stream);

/* ---- matrix products over a few rows, teal_amd/csrc/teal_rows.hip -----------------------------------------------------
 * y[M][N] = x[M][K] * W^T image [K][ld] for M <= 64, K % 32 == 0, N % 8 == 0, 16-bit operands, fp32 sums (over slices of K in slice order:
 * bit-reproducible).  x rows ldx apart (ldx % 8 == 0), ld % 8 == 0; x, images and biases 16-byte aligned. */
#define TEAL_ROWS_ROUNDED 0 /* y 16-bit [M][ldy] (ldy % 4 == 0) = round(act(sum + bias)), or with w_up round(act(sum + bias) * (sum_up + bias_up)) */
#define TEAL_ROWS_SLABS 1   /* y fp32 [teal_rows_split()][M][N]: the slices' partial sums, for the consumer to add in slice order */
#define TEAL_ROWS_F32 2     /* y fp32 [M][ldy], columns < n_valid: the sum, or softcap * tanh(sum / softcap) */
#define TEAL_ACT_NONE (-1)
#define TEAL_ACT_SILU_ROUNDED 3 /* with w_up: round(silu(round(gate))) * round(up), the rounding points of gpt-fast/model.py:258-259 */
typedef struct teal_rows_gemm {
    const void* x;
    const void* w;
    const void* w_up;          /* optional second image (same ld): gate = w, up = w_up */
    const void* bias;          /* optional, 16-bit [N] */
    const void* bias_up;
    void* y;
    float* part;               /* ROUNDED, F32 when teal_rows_split() > 1: scratch, split * M * (N rounded up to 128, with w_up 2 N to 128) floats */
    size_t part_bytes;
    unsigned* tickets;         /* ... and one zero counter per 128 (with w_up 64) columns, <= 256; zero again afterwards.  Launches that may
                                * overlap need their own */
    int M, K, N, ldx, ld, ldy;
    int mode, act, n_valid;
    float softcap;
} teal_rows_gemm_t;
/* slices a launch of this shape takes (>= 1); 0: outside the kernel's shapes */
int teal_rows_split(int M, int K, int N, int paired);
int teal_rows_gemm(const teal_rows_gemm_t* args, int dtype, void* stream);

/* ---- matrix products over a prompt's rows, teal_amd/csrc/teal_tile.hip -------------------------------------------------
 * The same product for any number of rows: x [M][ldx] times one W^T image [K][ld], or two of one shape (gate and up); K % 64 == 0, N % 16 == 0.
 * Results 16-bit y0 / y1 [M][ldy] (ldy % 8 == 0), or (slabs given, one image) the fp32 partial sums [teal_tile_split()][M][N]. */
/* slices of K such a launch takes (1 without slabs); 0: not a case for it (the shape, or a vendor library is faster) */
int teal_tile_split(int M, int K, int N, int images, int slabs);
int teal_tile_gemm(const void* x, int ldx, const void* w0, const void* w1, int ld, void* y0, void* y1, int ldy, float* slabs, int M, int K, int N, int dtype,
                   void* stream);

/* ---- layered decoder designs: row kernels around their matrix products, teal_amd/csrc/teal_layered.hip ----------------
 * dtype 0 / 1 / 2 (fp16, bf16, fp32) = activations and weights; the residual stream is always fp32. */

/* Per row r (= rows[i], or i): x[r] = embed[tokens[r]] | x[r], plus y[r] (+ y_bias) — RMS-normed with post_w first when post_w is
 * given — and then h[i] = x[r] / sqrt(mean(x[r]^2) + eps) * (norm_offset + pre_w) (rounded once; post_w alike).  tokens / y / post_w / pre_w are optional; h is
 * packed [n_rows][dim].  Token ids are clamped to the table.  dim <= 15360. */
int teal_layer_resid_norm(float* x, int n_rows, int dim, const int32_t* tokens, const void* embed, int vocab, const void* y, int ldy,
                          const void* y_bias, const void* post_w, const void* pre_w, float norm_offset, float eps, void* h,
                          const int32_t* rows, int dtype, void* stream);
/* the same with y = the sum of n_slabs fp32 slabs [n_slabs][n_rows][ldy] in slab order (TEAL_ROWS_SLABS; rows: indexes them too, of slab_rows
 * rows); zero: optional, n_zero <= 256 counters set to zero (the tickets of the products that follow) */
int teal_layer_resid_norm_slabs(float* x, int n_rows, int dim, const int32_t* tokens, const void* embed, int vocab, const float* y, int n_slabs, int slab_rows,
                                int ldy, const void* y_bias, const void* post_w, const void* pre_w, float norm_offset, float eps, void* h,
                                const int32_t* rows, unsigned* zero, int n_zero, int dtype, void* stream);
#define TEAL_ACT_SILU 0
#define TEAL_ACT_GELU_TANH 1
#define TEAL_ACT_RELU2 2 /* max(z, 0)^2 */
/* h[t][n] = act(gu[t][n] + bias_gate[n]) * (gu[t][up0 + n] + bias_up[n]), n < n_cols; the biases are optional; up0 = 0: no second factor */
int teal_gated_act(const void* gu, int ldg, int up0, const void* bias_gate, const void* bias_up, void* h, int ldh, int n_rows, int n_cols,
                   int act, int dtype, void* stream);
/* out (fp32 [n_rows][vocab]) = cap * tanh(logits / cap); cap <= 0: the conversion alone */
int teal_logit_softcap(const void* logits, int ld, float* out, int n_rows, int vocab, float cap, int dtype, void* stream);
/* One token per row of fp32 logits [n_rows][ld]: top-k filter (ties at the k-th stay; top_k <= 0 or >= vocab: none), softmax, exponential
 * race; temperature <= 0: the largest logit (the lowest index of equals).  rng_state = device uint64 [n_rows][2] {seed, draw counter},
 * bumped per draw; optional loop state: pos_inout[row] += 1, history[row][draw counter] = token. */
int teal_sample_rows(const float* logits, int ld, int n_rows, int vocab, int top_k, float temperature, void* rng_state, int32_t* token_out,
                     int32_t* pos_inout, int32_t* history, int history_len, void* stream);

/* ---- latent attention, teal_amd/csrc/teal_latent.hip -------------------------------------------------------------------
 * Sizes: heads; per head dim unrotated + rot rotated query / key dimensions and vdim value dimensions; rank = size of the latent.
 * proj rows: [q (heads x (dim + rot)) | ... | latent (rank), shared key part (rot) at column kv0]; kv0 < 0: the layer reads another
 * layer's cache and writes none.  Cache: rows of ldc elements [latent | rotated key part | padding], pages of 2^page_shift rows;
 * table [slots][max_pages] holds a sequence slot's page ids.  inv_freq [rot / 2]: angle of pair i at position p = p * inv_freq[i].
 * window: a query at p sees p - window < j <= p.  sink [heads], gate [..][heads * vdim] optional.  dtype 0 / 1 / 2. */

/* prompt pass: rotate the queries in place; write the cache row row[t] of every token (RMS-normed latent, rotated key part) */
int teal_latent_prompt_rows(void* proj, int ldp, int kv0, int n_tokens, const int32_t* pos, const int32_t* row, const float* inv_freq, const void* norm_w,
                            float eps, int heads, int dim, int rot, int rank, void* cache, int ldc, int dtype, void* stream);
/* packed copies c [n_rows][rank], kr [n_rows][rot] of cache rows row[i] (row[i] < 0: zeros) */
int teal_latent_gather(const void* cache, int ldc, const int32_t* row, int n_rows, int rank, int rot, void* c, void* kr, int dtype, void* stream);
/* queries per workgroup of the attention launch over prompts whose longest portion is n_queries (1: the scalar kernel) */
int teal_layer_prompt_tile(int dim, int rot, int vdim, int n_queries, int dtype);
/* attention over expanded keys k [n_keys][heads / group * dim], kr [n_keys][rot] and values vt [heads / group * vdim][n_keys] (n_keys % 8
 * == 0): query head h reads key / value head h / group.  softcap > 0 (with vdim <= dim + rot): scores become softcap * tanh(score / softcap).
 * seqs: int32 [..][5] = first query row, queries, position of the first query, packed key row of position klo (a multiple of 64,
 * every sequence's span padded to a multiple of 64), klo; tiles: int32 [n_tiles][2] = sequence, first query (a multiple of tile).
 * out [..][ldo] = attention output * sigmoid(gate). */
int teal_layer_prompt_attention(const void* q, int ldq, const void* k, const void* kr, const void* vt, int n_keys, const void* sink, const void* gate,
                                 int ldg, void* out, int ldo, const int32_t* seqs, const int32_t* tiles, int n_tiles, int tile, int heads, int group, int dim,
                                 int rot, int vdim, int window, float scale, float softcap, int dtype, void* stream);
/* one token per sequence: the absorbed, rotated query -> qcat [batch][heads][ldq] (fp32) or [batch][heads][2][ldq] (16-bit: high and
 * low halves), ldq % 32 == 0; the token's cache row at position pos[b] of slot[b].  uk [heads * dim][rank]. */
int teal_latent_step_query(const void* proj, int ldp, int kv0, int batch, const int32_t* pos, const int32_t* slot, const int32_t* table, int max_pages, int page_shift,
                           const float* inv_freq, const void* norm_w, float eps, const void* uk, int heads, int dim, int rot, int rank, void* cache, int ldc, void* qcat,
                           int ldq, int dtype, void* stream);
/* ... partial attention over the cached rows of the window, split over `splits` workgroups per 16 heads; a cached row of ldc elements
 * holds heads / group segments of ldq elements, each shared by `group` heads (latent attention: one segment, ldc = ldq):
 * part fp32 [batch][heads][splits][R4 + 4], R4 = rank rounded up to 4: {weighted latent [R4], max of the scaled scores in log2
 * units, sum, -, -} */
int teal_layer_step_attention(const void* qcat, int ldq, const void* cache, int ldc, const int32_t* pos, const int32_t* slot, const int32_t* table, int max_pages,
                              int page_shift, int batch, int heads, int group, int rank, int rot, int window, float scale, float softcap, int splits, float* part,
                              size_t part_bytes, int dtype, void* stream);
/* ... and y [batch][ldy] = (W_uv,head (merged latent)) * sigmoid(gate); uv [heads * vdim][rank] */
int teal_latent_step_merge(const float* part, int splits, const void* uv, const void* sink, const void* gate, int ldg, void* y, int ldy, int batch, int heads, int rank,
                           int vdim, int dtype, void* stream);

/* ---- grouped-query attention over tied keys and values (a value is its key before rotation), teal_amd/csrc/teal_grouped.hip --------
 * proj rows: [queries (heads x dim) | ... | keys (kv_heads x dim) at column k0].  Cache rows: kv_heads segments of ldk elements [key (dim) |
 * its first rot dimensions, rotated | zeros], ldk % 32 == 0.  A prompt's attention launch is teal_layer_prompt_attention (dim, rot = 0, vdim =
 * dim, the gathered keys). */
int teal_grouped_prompt_rows(void* proj, int ldp, int k0, int n_tokens, const int32_t* pos, const int32_t* row, const float* inv_freq, int heads, int kv_heads, int dim,
                             int rot, void* cache, int ldk, int dtype, void* stream);
/* k [n_rows][kv_heads][dim] (rotated), vt [kv_heads * dim][n_rows] of cache rows row[i] (row[i] < 0: zeros) */
int teal_grouped_gather(const void* cache, int ldk, const int32_t* row, int n_rows, int kv_heads, int dim, int rot, void* k, void* vt, int dtype, void* stream);
/* one token per sequence: the token's cache row and the partial attention over the window, part as teal_layer_step_attention's (rank =
 * dim).  One launch over the matrix cores; 32-bit elements and sizes beyond them: the two launches it is made of, the query rows in
 * qcat [batch][heads][ldk] (16-bit: [2][ldk]; else not used) */
int teal_grouped_step_attention(const void* proj, int ldp, int k0, int batch, const int32_t* pos, const int32_t* slot, const int32_t* table, int max_pages, int page_shift,
                                const float* inv_freq, int heads, int kv_heads, int dim, int rot, void* cache, int ldk, int window, float scale, float softcap, int splits,
                                void* qcat, float* part, size_t part_bytes, int dtype, void* stream);
int teal_grouped_step_query(const void* proj, int ldp, int k0, int batch, const int32_t* pos, const int32_t* slot, const int32_t* table, int max_pages, int page_shift,
                            const float* inv_freq, int heads, int kv_heads, int dim, int rot, void* cache, int ldk, void* qcat, int ldq, int dtype, void* stream);
/* y [batch][ldy] = merged splits (sink [heads] optional) */
int teal_grouped_step_merge(const float* part, int splits, const void* sink, void* y, int ldy, int batch, int heads, int dim, int dtype, void* stream);

/* ---- time mixing with a decaying matrix state, teal_amd/csrc/teal_wkv.hip ---------------------------------------------
 * Per sequence slot and layer: shift rows fp32 [slots][2][width], states fp32 [slots][2][heads][dim (key)][dim (value)]; the token at
 * position p reads buffer (p - 1) & 1 (zeros at p = 0) and writes buffer p & 1, so a repeated step repeats its result.  dim <= 256. */

/* out [n_mix][n_rows][dim]: h + (previous h - h) * mu[s], h = RMSNorm(x) * (norm_offset + norm_w) in fp32.  run[t] > 0 marks the first row
 * of a portion of run[t] rows (its predecessor comes from the state, its last row goes there), null: every row is a portion. */
int teal_wkv_mix(const float* x, int n_rows, int dim, const void* norm_w, float norm_offset, float eps, const void* mu, int n_mix, const int32_t* pos,
                 const int32_t* slot, const int32_t* run, float* state, void* out, int dtype, void* stream);
/* out [n_rows][channels] = exp(-exp(w2 tanh(z) + w0)); z [n_rows][ldz], w2 [channels][rank], rank <= 512 */
int teal_wkv_decay(const void* z, int ldz, const void* w2, const void* w0, int rank, int n_rows, int channels, float* out, int dtype, void* stream);
/* the recurrence over the portions seqs [..][5] (first row, rows, position of the first row, -, -), the longest of them `longest` rows; w =
 * decays, u [heads][dim], o fp32 [n_rows][heads * dim].  `chunks`: scratch of teal_wkv_chunk_bytes.  Two launches. */
size_t teal_wkv_chunk_bytes(int n_rows, int n_seqs, int heads, int dim);
int teal_wkv_scan(const void* r, const void* k, const void* v, int ldp, const float* w, const void* u, const int32_t* seqs, int n_seqs, int n_rows, int longest,
                  const int32_t* slot, float* state, float* chunks, size_t chunk_bytes, float* o, int heads, int dim, int dtype, void* stream);
/* y = o / rms of its head * norm * silu(g) */
int teal_wkv_out(const float* o, const void* norm, const void* g, int ldg, float eps, void* y, int ldy, int n_rows, int heads, int dim, int dtype, void* stream);
/* one token per sequence, from the projections to y: decay, recurrence, state update, head norm and gate */
int teal_wkv_step(const void* r, const void* k, const void* v, const void* g, int ldp, const void* z, int ldz, const void* w2, const void* w0, int rank, const void* u,
                  const void* norm, float eps, const int32_t* pos, const int32_t* slot, float* state, void* y, int ldy, int batch, int heads, int dim, int dtype,
                  void* stream);

/* ---- benchmark comparator (scripts/benchmark_gemv.py only; not on the decode path) ----------- */

/* The Deja Vu gather GEMV the reference's kernel benchmark plots next to TEAL's (scripts/benchmark_gemv.py:32-107,170-172),
 * restated for CDNA4: flags[m] = |x[m]| > tau by a launch of its own, y32 zeroed, then a (row block, column tile) grid adds
 * fp32 partial sums of the flagged rows into y32 with atomics.  y32: fp32 [N]; flags: Z bytes of scratch.  Three launches. */
int teal_cmp_flag_gemv(const void* x, const void* wT, int ld, float* y32, unsigned char* flags, float tau, int Z, int N,
                       int dtype, void* stream);

/* ---- diagnostics build only (libteal_hip_diag.so = these sources with -DTEAL_DIAGNOSTICS) ------------------------
 * Process-global switches, NOT thread-safe, for benchmarks, phase-stamp probes and the parity tests that force the general
 * kernel or a launch geometry.  libteal_hip.so exports none of them. */
#ifdef TEAL_DIAGNOSTICS

/* Override the launch geometry picked from (Z, N, CU count): lanes per row segment (8/16/32/64) and split-K factor
 * (>= 1); waves per workgroup and unroll depth are fixed at 16 and 4 (the other values of round 1 were sweep-only
 * and are no longer built: pass 0 or the fixed value).  0 = automatic.  Process-global; meant for benchmark sweeps only. */
int teal_set_tuning(int lanes_per_row, int waves, int split, int unroll);

/* Wave-local compaction (default on): each wave streams the rows it ballots itself instead of an even share
 * of a workgroup-wide list; removes every barrier between the activation and the first weight load. */
int teal_set_wave_local(int on);

/* Diagnostics: kernel template instantiation and grid of the most recent GEMV launch of this process (host-side
 * string; e.g. for naming the kernel in a benchmark record). */
const char* teal_last_launch_desc(void);

/* Lean kernel for qualifying shapes (default on; 0 forces the general kernel everywhere: A/B and parity tests). */
int teal_set_fast(int on);

/* Diagnostics: when set (device pointer to >= 32 * workgroups uint64 — 32 stamps per workgroup of the launch), every
 * GEMV workgroup stores 100 MHz wall-clock stamps of its phases, row w of the buffer = workgroup w:
 *   [0] kernel entry, [1] kernel arguments in registers, [2] activation ready, [3] row list ready, [4] first weight
 *   batch consumed (wave 0), [5] wave 0 done streaming, [6] past the reduce barrier, [7] done,
 *   [12] hardware id << 32 | XCC id, [13] waves << 32 | workgroups, [16 + w] end of stream of wave w (w < 16).
 * The attention, sampler and int4 launches (the latter with fp16 activations only) stamp rows of the same width with their own
 * phase meanings (scripts/attn_phase.py, scripts/sampler_phase.py, scripts/int4_phase.py).  NULL (default) disables.
 * Process-global. */
int teal_set_phase_buffer(void* dev_u64);
/* > 0: consecutive GEMV / attention launches stamp consecutive regions of `u64_per_launch` uint64 of the phase buffer
 * (so that a chain of launches can be timed against each other): u64_per_launch >= 32 * the largest launch's
 * workgroups, and the buffer must hold u64_per_launch * (launches between two teal_set_phase_stride calls) uint64;
 * 0 (default): every launch stamps the start of the buffer. */
int teal_set_phase_stride(size_t u64_per_launch);
#endif /* TEAL_DIAGNOSTICS */

/* ---- introspection (pure function of its arguments and the device's CU count) ------------------ */

/* The geometry a GEMV of this shape would use: out[0..5) = {lanes_per_row, waves, split, unroll,
 * workgroups}. */
int teal_get_config(int Z, int N, int nseg, int* out);

#ifdef __cplusplus
}
#endif
#endif /* TEAL_HIP_H */
