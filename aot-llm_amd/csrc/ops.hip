// ops.hip - the non-matmul operators of the transformer block on gfx950
// (crates/aot-kernels/src/ops.rs), fused with the activation quantization
// that follows each of them in the generated forward (emit.rs:243-333):
//   rmsnorm -> quantize_q8_k / q8_0, silu_mul / gelu_mul -> quantize,
//   bias + rmsnorm_heads + rope + store_kv in one per-head kernel,
//   GQA decode attention split over position chunks (K/V rows read once),
//   argmax over the vocabulary.
// Every float sum that feeds an activation quantizer runs in the reference's
// sequential order (a different order changes results by an ulp, which flips
// int8 roundings downstream); transcendental functions are the host-libm
// matched aotk_expf / aotk_tanhf. Maxima and integer sums use trees.
#include <algorithm>

#include "device.hpp"
#include "lds_chain.hpp"
#include "formats.hpp"
#include "internal.hpp"
#include "seqsum.hpp"
#include "actfn.hpp"

namespace aotk {

__device__ __forceinline__ float wave_sum(float v) {
    for (int m = 1; m < 64; m <<= 1) v += shfl_xor(v, m);
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
    for (int m = 1; m < 64; m <<= 1) v = fmaxf(v, shfl_xor(v, m));
    return v;
}

// Block-wide sum (blockDim.x multiple of 64, at most 1024). Same tree for
// every call with the same blockDim, so results are reproducible.
__device__ float block_sum(float v, float *red) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    v = wave_sum(v);
    __syncthreads();
    if (lane == 0) red[wave] = v;
    __syncthreads();
    float t = lane < nw ? red[lane] : 0.0f;
    t = wave_sum(t);
    return t;
}

// Sequential f32 sum of n LDS values in index order, by one thread: v 16-byte
// aligned and padded with -0.0 up to a multiple of 64 values.
__device__ __forceinline__ float seq_sum_lds_pad64(const float *v, int n) {
    return lds_chain(v, (n + 63) >> 6, 0.0f);
}

// ss = sum of v*v over n <= 256 values in LDS, in index order
// (ops.rs:10-13), for one wave: the lanes form the squares (each rounded as
// in the sequential loop) into tmp, padded with -0.0 to a run of 64 (neutral
// under round to nearest), then lane 0 adds them in order with the LDS
// chain; the result is returned to every lane.
__device__ __forceinline__ float wave_sumsq_lds(const float *v, float *tmp, int n) {
    const int lane = threadIdx.x & 63;
    const int n64 = (n + 63) & ~63;
    for (int e = lane; e < n64; e += 64) tmp[e] = e < n ? v[e] * v[e] : -0.0f;
    wave_lds_sync();
    float ss = 0.0f;
    if (lane == 0) ss = seq_sum_lds_pad64(tmp, n);
    return __shfl(ss, 0, 64);
}

__device__ __forceinline__ ActQ8K q8k_row(ActQ8K a, size_t row, size_t n) {
    if (!a.qs) return a;
    ActQ8K r = a;
    r.qs += row * n;
    r.d += row * (n / 256);
    r.bsums += row * (n / 16);
    r.tok = (int)row;
    r.nbt = (int)(n / 256);
    return r;
}
__device__ __forceinline__ ActQ8_0 q80_row(ActQ8_0 a, size_t row, size_t n) {
    if (!a.qs) return a;
    ActQ8_0 r = a;
    r.qs += row * n;
    r.d += row * (n / 32);
    r.tok = (int)row;
    r.nbt = (int)(n / 32);
    return r;
}

// rmsnorm (ops.rs:7-18) of row blockIdx.x, then quantization of the result.
// n % 256 == 0, n <= 8192 (the normalised row is staged in LDS).
#ifndef RMS_TS
#define RMS_TS(i)
#endif
__global__ __launch_bounds__(SEQ_T) void k_rmsnorm_quant(const float *__restrict__ x, const float *__restrict__ w, int n,
                                                         float eps, RmsOut out) {
    __shared__ __align__(16) float row[8192];
    __shared__ float sq[SEQ_PAD_N];
    __shared__ SeqScratch S;
    const size_t m = blockIdx.x;
    const float *xr = x + m * n;
    const int C = seq_chunk(n);
    RMS_TS(0);
    // all of a thread's loads are in flight together (n <= 8 * blockDim.x):
    // the row first, then the norm weights, which stay in flight during the
    // sum (the loads complete in order, so the squares wait for the row only)
    float xv[8], wv[8];
#pragma unroll
    for (int k = 0; k < 8; k++) xv[k] = xr[min((int)threadIdx.x + k * SEQ_T, n - 1)];
#pragma unroll
    for (int k = 0; k < 8; k++) wv[k] = w[min((int)threadIdx.x + k * SEQ_T, n - 1)];
    // the row is needed here, on every path: no load may move into the
    // conditional stores below (and wait there for the norm weights)
#pragma unroll
    for (int k = 0; k < 8; k++) asm volatile("" : "+v"(xv[k]));
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int i = threadIdx.x + k * SEQ_T;
        if (i < n) {
            row[i] = xv[k];
            sq[seq_idx(i, C)] = xv[k] * xv[k];
        }
    }
    __syncthreads();
    RMS_TS(1);
    float ss = exact_seq_sum(sq, n, S);
    RMS_TS(2);
    float r = 1.0f / sqrtf(ss / (float)n + eps);
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int i = threadIdx.x + k * SEQ_T;
        if (i < n) {
            const float v = row[i] * r * wv[k];
            row[i] = v;
            if (out.f32) out.f32[m * n + i] = v;
        }
    }
    RMS_TS(4);
    __syncthreads();
    RMS_TS(5);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    ActQ8K qk = q8k_row(out.q8k, m, n);
    ActQ8_0 q0 = q80_row(out.q80, m, n);
    for (int b = wave; b < n / 256; b += nw) {
        float4 v4 = ((const float4 *)(row + b * 256))[lane];
        float v[4] = {v4.x, v4.y, v4.z, v4.w};
        quant256(v, lane, b, qk, q0);
    }
    RMS_TS(3);
}

// Rows of whole 256-value blocks: thread t holds float4 t (+ 1024 k) of the
// row, so wave w holds the values of quantization blocks w (+ 16 k) in
// quant256's lane order: the normalised row goes from registers straight
// to the quantizer, with no LDS copy and no barrier after the sum.
template <int KF>
__global__ __launch_bounds__(SEQ_T) void k_rmsnorm_quant4(const float *__restrict__ x, const float *__restrict__ w, int n,
                                                         float eps, RmsOut out) {
    __shared__ float sq[SEQ_PAD_N];
    __shared__ SeqScratch S;
    const size_t m = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63;
    const int n4 = n / 4;
    const int C = seq_chunk(n);
    const float4 *xr = (const float4 *)(x + m * n);
    RMS_TS(0);
    float4 xv[KF], wv[KF];
#pragma unroll
    for (int k = 0; k < KF; k++) {
        const int i = tid + k * SEQ_T;
        xv[k] = i < n4 ? xr[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
#pragma unroll
    for (int k = 0; k < KF; k++) {
        const int i = tid + k * SEQ_T;
        wv[k] = i < n4 ? ((const float4 *)w)[i] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
#pragma unroll
    for (int k = 0; k < KF; k++) {
        const int i = tid + k * SEQ_T;
        if (i < n4) {
            sq[seq_idx(4 * i, C)] = xv[k].x * xv[k].x;
            sq[seq_idx(4 * i + 1, C)] = xv[k].y * xv[k].y;
            sq[seq_idx(4 * i + 2, C)] = xv[k].z * xv[k].z;
            sq[seq_idx(4 * i + 3, C)] = xv[k].w * xv[k].w;
        }
    }
    __syncthreads();
    RMS_TS(1);
    const float ss = exact_seq_sum(sq, n, S);
    RMS_TS(2);
    const float r = 1.0f / sqrtf(ss / (float)n + eps);
    const ActQ8K qk = q8k_row(out.q8k, m, n);
    const ActQ8_0 q0 = q80_row(out.q80, m, n);
#pragma unroll
    for (int k = 0; k < KF; k++) {
        const int i = tid + k * SEQ_T;
        if (i < n4) {  // wave-uniform: n4 is a multiple of 64
            const float v[4] = {xv[k].x * r * wv[k].x, xv[k].y * r * wv[k].y, xv[k].z * r * wv[k].z, xv[k].w * r * wv[k].w};
            if (out.f32) *(float4 *)(out.f32 + m * n + 4 * i) = make_float4(v[0], v[1], v[2], v[3]);
            quant256(v, lane, (size_t)(i >> 6), qk, q0);
        }
    }
    RMS_TS(3);
}

void launch_rmsnorm_quant(const float *x, const float *w, size_t n, size_t m, float eps, RmsOut out, hipStream_t s) {
    if (m < 2) out.q8k.qt = nullptr, out.q80.xh = nullptr;  // the tiled / f16 copies serve batches only
    if (n % 256 == 0 && n <= 4096) k_rmsnorm_quant4<1><<<(unsigned)m, SEQ_T, 0, s>>>(x, w, (int)n, eps, out);
    else if (n % 256 == 0) k_rmsnorm_quant4<2><<<(unsigned)m, SEQ_T, 0, s>>>(x, w, (int)n, eps, out);
    else k_rmsnorm_quant<<<(unsigned)m, SEQ_T, 0, s>>>(x, w, (int)n, eps, out);
}

// Quantize m rows of n floats (n % 256 == 0), one wave per 256 values.
__global__ void k_quant_f32(const float *__restrict__ x, int n, size_t total_blk, RmsOut out) {
    const int lane = threadIdx.x & 63;
    size_t gb = (size_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (gb >= total_blk) return;
    size_t per = (size_t)n / 256;
    size_t m = gb / per, b = gb % per;
    float4 v4 = ((const float4 *)(x + m * n + b * 256))[lane];
    float v[4] = {v4.x, v4.y, v4.z, v4.w};
    quant256(v, lane, b, q8k_row(out.q8k, m, n), q80_row(out.q80, m, n));
}

void launch_quant_f32(const float *x, size_t n, size_t m, RmsOut out, hipStream_t s) {
    if (m < 2) out.q8k.qt = nullptr, out.q80.xh = nullptr;  // the tiled / f16 copies serve batches only
    size_t total = m * n / 256;
    k_quant_f32<<<(unsigned)((total + 3) / 4), 256, 0, s>>>(x, (int)n, total, out);
}

// silu_mul / gelu_mul (ops.rs:115-134) then quantization: block = one
// quantization block of 256 values, one value per thread (the libm-matched
// exp / tanh run once per lane, not four times in a row), then wave 0
// quantizes the block from LDS.
__global__ __launch_bounds__(256) void k_glu_quant(const float *__restrict__ gate, const float *__restrict__ up, int n,
                                                   size_t total_blk, int gelu, RmsOut out) {
    __shared__ __align__(16) float sv[256];
    const size_t gb = blockIdx.x;
    if (gb >= total_blk) return;
    const int t = threadIdx.x;
    const size_t per = (size_t)n / 256;
    const size_t m = gb / per, b = gb % per;
    const size_t off = m * n + b * 256 + t;
    const float g = gate[off], u = up[off];
    const float v = gelu ? gelu_f(g) * u : silu_f(g, u);
    sv[t] = v;
    if (out.f32) out.f32[off] = v;
    __syncthreads();
    if (t < 64) {
        const float4 v4 = ((const float4 *)sv)[t];
        float vv[4] = {v4.x, v4.y, v4.z, v4.w};
        quant256(vv, t, b, q8k_row(out.q8k, m, n), q80_row(out.q80, m, n));
    }
}

void launch_glu_quant(const float *gate, const float *up, size_t n, size_t m, int gelu, RmsOut out, hipStream_t s) {
    if (m < 2) out.q8k.qt = nullptr, out.q80.xh = nullptr;  // the tiled / f16 copies serve batches only
    size_t total = m * n / 256;
    k_glu_quant<<<(unsigned)total, 256, 0, s>>>(gate, up, (int)n, total, gelu, out);
}

// Embedding rows (dequant_row of the token's row, emit.rs:469) [* sqrt(dim)].
template <int KIND>
__global__ void k_embed(WView w, const uint32_t *__restrict__ tokens, size_t cols, float scale, int do_scale, float *x) {
    size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    size_t i = blockIdx.y;
    if (c >= cols) return;
    float v = dequant_elem<KIND>(w, tokens[i], c);
    if (do_scale) v = v * scale;
    x[i * cols + c] = v;
}

void launch_embed(const DevWeight &embd, const uint32_t *tokens, size_t m, float scale, int do_scale, float *x, hipStream_t s) {
    dim3 grid((unsigned)((embd.cols + 255) / 256), (unsigned)m);
    WView v = view_of(embd);
#define F(K) k_embed<K><<<grid, 256, 0, s>>>(v, tokens, embd.cols, scale, do_scale, x)
    AOTK_KIND_SWITCH(embd.kind, F)
#undef F
}

// ------------------------------------------------ q/k/v per-head epilogue
// One wave per (row, head): bias (ops.rs:89-95), rmsnorm_heads (ops.rs:74-87),
// rope / rope_neox (ops.rs:40-70) with the row's position table, and the
// store_kv copy into the cache (ops.rs:152-157). Heads [0, n_head) are q,
// [n_head, n_head + n_kv_head) are k (+ v).
__global__ __launch_bounds__(64) void k_qkv_post(QkvPost p, size_t pos0, const int *pos_dev) {
    __shared__ __align__(16) float hv[256];
    const int lane = threadIdx.x;
    const size_t i = blockIdx.y;
    const int hh = blockIdx.x;
    const bool is_q = hh < (int)p.n_head;
    const int h = is_q ? hh : hh - (int)p.n_head;
    const int hd = (int)p.head_dim;
    const size_t q_dim = p.n_head * hd, kv_dim = p.n_kv_head * hd;
    const size_t pos = pos_dev ? (size_t)*pos_dev : pos0 + i;
    float *vec = is_q ? p.q + i * q_dim + (size_t)h * hd : p.k + i * kv_dim + (size_t)h * hd;
    const float *bias = is_q ? p.bq : p.bk;
    const float *nw = is_q ? p.q_norm : p.k_norm;
    for (int e = lane; e < hd; e += 64) {
        float v = vec[e];
        if (bias) v = v + bias[(size_t)h * hd + e];
        hv[e] = v;
    }
    __syncthreads();
    if (nw) {
        __shared__ __align__(16) float sqt[256];
        float ss = wave_sumsq_lds(hv, sqt, hd);
        float r = 1.0f / sqrtf(ss / (float)hd + p.eps);
        for (int e = lane; e < hd; e += 64) hv[e] = hv[e] * r * nw[e];
        __syncthreads();
    }
    const float *cs = p.cs + pos * p.rot_dim;
    const int half = (int)p.rot_dim / 2;
    for (int t = lane; t < half; t += 64) {
        float c = cs[2 * t], s = cs[2 * t + 1];
        int a = p.neox ? t : 2 * t, b = p.neox ? t + half : 2 * t + 1;
        float x0 = hv[a], x1 = hv[b];
        hv[a] = x0 * c - x1 * s;
        hv[b] = x0 * s + x1 * c;
    }
    __syncthreads();
    for (int e = lane; e < hd; e += 64) vec[e] = hv[e];
    if (!is_q) {
        float *kc = p.k_cache + pos * kv_dim + (size_t)h * hd;
        float *vc = p.v_cache + pos * kv_dim + (size_t)h * hd;
        const float *vsrc = p.v + i * kv_dim + (size_t)h * hd;
        for (int e = lane; e < hd; e += 64) {
            kc[e] = hv[e];
            float v = vsrc[e];
            if (p.bv) {
                v = v + p.bv[(size_t)h * hd + e];
                ((float *)vsrc)[e] = v;
            }
            vc[e] = v;
        }
    }
}

void launch_qkv_post(const QkvPost &p, size_t m, size_t pos0, const int *pos_dev, hipStream_t s) {
    dim3 grid((unsigned)(p.n_head + p.n_kv_head), (unsigned)m);
    k_qkv_post<<<grid, 64, 0, s>>>(p, pos0, pos_dev);
}

// ----------------------------------------------------------- attention
// Causal GQA attention (ops.rs:185-218 `attention`, :517-556
// `attention_rows`) in the reference's arithmetic order, in three passes:
//   1. scores: one thread per cached position computes q.k sequentially over
//      the head dimension for every query head of the kv group (each K row is
//      read once for the group), times 1/sqrt(hd);
//   2. softmax per (row, head): max, host-libm exp, a sequential sum in
//      position order, multiply by 1/sum (ops.rs:98-112);
//   3. output: one thread per (head, dim) accumulates p_t * v_t in position
//      order (ops.rs:209-215); V rows are read coalesced across dims.
// Scratch: probabilities [m][n_head][span].
constexpr int ATT_CH = 64;
constexpr int ATT_MAX_GQA = 8;

struct AttnArgs {
    float *out;
    const float *q, *k_cache, *v_cache;
    float *prob;
    int n_head, n_kv_head, hd, span;
    size_t pos0, window;
    const int *pos_dev;
    float scale;
};

__device__ __forceinline__ void row_range(const AttnArgs &a, size_t i, size_t &t0, size_t &n) {
    size_t pos = a.pos_dev ? (size_t)*a.pos_dev : a.pos0 + i;
    n = pos + 1;
    t0 = (a.window > 0 && pos + 1 > a.window) ? pos + 1 - a.window : 0;
}

// Scores of one row: block = (kv head, chunk of ATT_CH positions), gqa * 64
// threads. The chunk's K rows are staged in LDS (coalesced row loads, eight per
// thread in flight; row stride HD + 4: 16-byte rows, the 16-byte reads of 16
// rows hit all banks); thread (query head of the group, position) then runs its
// dot product sequentially over the head dimension. 8 kv heads x 4100
// positions, head_dim 128 (16.8 MB): 8.0 -> 6.7 us against one load at a time
// and 4-byte reads.
template <int HD>
__global__ __launch_bounds__(512) void k_attn_scores(AttnArgs a) {
    constexpr int KS = HD + 4;
    __shared__ __align__(16) float sk[ATT_CH * KS];
    __shared__ __align__(16) float sq[ATT_MAX_GQA][HD];
    const int gqa = a.n_head / a.n_kv_head;
    const int lane = threadIdx.x & 63, hg = threadIdx.x >> 6;
    const int kvh = blockIdx.x, c = blockIdx.y;
    size_t t0, n;
    row_range(a, 0, t0, n);
    const size_t start = t0 + (size_t)c * ATT_CH;
    if (start >= n) return;
    const int rows = (int)min((size_t)ATT_CH, n - start);
    const size_t kv = (size_t)a.n_kv_head * HD;
    const float *kb = a.k_cache + start * kv + (size_t)kvh * HD;
    constexpr int R4 = HD / 4;
    const int last = rows * R4 - 1, nth = (int)blockDim.x;
    const float *qs = a.q + (size_t)(kvh * gqa + hg) * HD;
    float qv[HD / 64];
#pragma unroll
    for (int j = 0; j < HD / 64; j++) qv[j] = qs[lane + 64 * j];
    for (int i0 = threadIdx.x; i0 <= last; i0 += 8 * nth) {
        float4 k4[8];  // (past the end: the last piece again, stored where it is)
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int idx = min(i0 + j * nth, last);
            k4[j] = *(const float4 *)(kb + (size_t)(idx / R4) * kv + 4 * (idx % R4));
        }
#pragma unroll
        for (int j = 0; j < 8; j++) {
            const int idx = min(i0 + j * nth, last);
            *(float4 *)(sk + idx / R4 * KS + 4 * (idx % R4)) = k4[j];
        }
    }
#pragma unroll
    for (int j = 0; j < HD / 64; j++) sq[hg][lane + 64 * j] = qv[j];
    __syncthreads();
    if (lane >= rows) return;
    const float4 *kr = (const float4 *)(sk + lane * KS);
    const float4 *qq = (const float4 *)sq[hg];
    float s = 0.0f;
#pragma unroll 8
    for (int d4 = 0; d4 < HD / 4; d4++) {
        const float4 k4 = kr[d4], q4 = qq[d4];
        s += q4.x * k4.x;
        s += q4.y * k4.y;
        s += q4.z * k4.z;
        s += q4.w * k4.w;
    }
    a.prob[(size_t)(kvh * gqa + hg) * a.span + (start + lane - t0)] = s * a.scale;
}

// Products of 16 steps for four rows at once: v_mfma_f32_4x4x1_f32 with a
// zero accumulator is one rounded product per output, x[row i] of step K
// (held by lane 4K + i of the register `x`, broadcast to every lane's block)
// times the lane's y[K]. Matrix and vector f32 take the same time per
// product, but the row operand needs no register copy per lane: a broadcast
// from LDS costs LDS bandwidth, and a DPP or scalar operand halves the
// multiply's rate (4.6 against 2.5 clocks). A sum started at +0 is never -0,
// so that the product's zero may lose its sign.
typedef float att_f4 __attribute__((ext_vector_type(4)));
template <int K = 0>
__device__ __forceinline__ void att_prod16(att_f4 (&p)[16], float x, const float (&y)[16]) {
    p[K] = __builtin_amdgcn_mfma_f32_4x4x1f32(x, y[K], att_f4{0.0f, 0.0f, 0.0f, 0.0f}, 4, K, 0);
    if constexpr (K + 1 < 16) att_prod16<K + 1>(p, x, y);
}

// Prompt scores: block = (kv head, chunk of 64 absolute positions, row
// group), wave = (query head, 4 RQ rows), lane = position. The chunk's K rows
// are staged in LDS once for the block (128 dimensions at a time); a lane
// reads its own row 16 bytes at a time and runs the rows' dot products side
// by side, each in dimension order: products by att_prod16, one add per
// (row, position, dimension) on the VALU, which bounds it (with q broadcast
// from LDS the reads did: 100 us at 64 rows x 32 heads x 4032 positions,
// head_dim 128).
template <int HD, int RQ>
__global__ __launch_bounds__(512) void k_attn_scores_rows(AttnArgs a, int m, int rgs) {
    constexpr int DC = HD < 128 ? HD : 128, KS = DC + 4, R = 4 * RQ;
    __shared__ __align__(16) float sk[ATT_CH * KS];
    const int gqa = a.n_head / a.n_kv_head;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kvh = blockIdx.x, h = kvh * gqa + wave % gqa;
    const size_t start = (size_t)blockIdx.y * ATT_CH;
    const int b0 = blockIdx.z * R * rgs, i0 = b0 + wave / gqa * R;
    // (rows' ranges move forward with the row)
    size_t lo, hi, tmp;
    row_range(a, (size_t)b0, lo, tmp);
    row_range(a, (size_t)min(b0 + R * rgs, m) - 1, tmp, hi);
    if (start >= hi || start + ATT_CH <= lo) return;  // no row has a position here
    const size_t kv = (size_t)a.n_kv_head * HD, q_dim = (size_t)a.n_head * HD;
    const float *kb = a.k_cache + (size_t)kvh * HD;
    const float *qp[RQ];  // lane 4b + i: dimension b of row i
#pragma unroll
    for (int r = 0; r < RQ; r++) qp[r] = a.q + (size_t)min(i0 + 4 * r + (lane & 3), m - 1) * q_dim + (size_t)h * HD + (lane >> 2);
    float q[RQ][HD / 16];
#pragma unroll
    for (int r = 0; r < RQ; r++)
#pragma unroll
        for (int g = 0; g < HD / 16; g++) q[r][g] = qp[r][16 * g];
    float s[RQ][4];
#pragma unroll
    for (int r = 0; r < RQ; r++) s[r][0] = s[r][1] = s[r][2] = s[r][3] = 0.0f;
#pragma unroll
    for (int c = 0; c < HD; c += DC) {
        if (c) __syncthreads();
        for (int idx = threadIdx.x; idx < ATT_CH * (DC / 4); idx += blockDim.x) {
            const int r = idx / (DC / 4), c4 = idx % (DC / 4);
            *(float4 *)(sk + r * KS + 4 * c4) = *(const float4 *)(kb + min(start + r, hi - 1) * kv + c + 4 * c4);
        }
        __syncthreads();
#pragma unroll
        for (int g = 0; g < DC / 16; g++) {
            float k[16];
#pragma unroll
            for (int j = 0; j < 4; j++) *(float4 *)&k[4 * j] = *(const float4 *)(sk + lane * KS + 16 * g + 4 * j);
#pragma unroll
            for (int r = 0; r < RQ; r++) {
                att_f4 p[16];
                att_prod16(p, q[r][c / 16 + g], k);
#pragma unroll
                for (int d = 0; d < 16; d++)
#pragma unroll
                    for (int i = 0; i < 4; i++) s[r][i] += p[d][i];
#pragma unroll
                for (int i = 0; i < 4; i++) asm volatile("" : "+v"(s[r][i]));  // (the adds here: sunk, the products would stay in registers)
            }
        }
    }
    const size_t t = start + lane;
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (i0 + r >= m) break;
        size_t t0, n;
        row_range(a, (size_t)(i0 + r), t0, n);
        if (t >= t0 && t < n) a.prob[((size_t)(i0 + r) * a.n_head + h) * a.span + (t - t0)] = s[r / 4][r % 4] * a.scale;
    }
}

// One wave's share of the q/k/v epilogue for one head vector (decode):
// bias, rmsnorm_heads (sequential sum of squares by lane 0), rope with the
// position's table row; the result is left in `hv` (LDS, HD floats). The
// inputs (the vector, its bias, the norm weights, the rope row) are loaded
// by head_load first, so that loads the caller issues afterwards (the K rows
// of the chunk) do not delay them.
template <int HD>
struct HeadIn {
    static constexpr int NE = (HD + 63) / 64;
    float v[NE], bv[NE], wv[NE];
    float2 cs[NE];
};
template <int HD>
__device__ __forceinline__ void head_load(HeadIn<HD> &in, const float *src, const float *bias, const float *nw,
                                          const float *cs_row, int rot_dim) {
    // unconditional loads (absent inputs read the vector itself, indices
    // past the end repeat the last element): no branch, so no wait, between
    // them
    const int lane = threadIdx.x & 63;
    const int half = rot_dim / 2;
    const float *bp = bias ? bias : src, *wp = nw ? nw : src;
    const float2 *cp = (const float2 *)cs_row;
#pragma unroll
    for (int k = 0; k < HeadIn<HD>::NE; k++) {
        const int e = min(lane + 64 * k, HD - 1);
        in.v[k] = src[e];
        in.bv[k] = bp[e];
        in.wv[k] = wp[e];
        in.cs[k] = cp[max(min(lane + 64 * k, half - 1), 0)];  // (rot_dim > 0 on this path)
    }
}
#ifndef EPI_TS
#define EPI_TS(i)
#endif
template <int HD>
__device__ __forceinline__ void head_post_wave(float *hv, float *tmp, const HeadIn<HD> &in, bool bias, bool norm,
                                               int rot_dim, int neox, float eps) {
    constexpr int NE = HeadIn<HD>::NE;
    const int lane = threadIdx.x & 63;
    const int half = rot_dim / 2;
#pragma unroll
    for (int k = 0; k < NE; k++) {
        const int e = lane + 64 * k;
        if (e < HD) hv[e] = bias ? in.v[k] + in.bv[k] : in.v[k];
    }
    wave_lds_sync();
    EPI_TS(4);
    if (norm) {
        const float ss = wave_sumsq_lds(hv, tmp, HD);
        EPI_TS(5);
        const float r = 1.0f / sqrtf(ss / (float)HD + eps);
#pragma unroll
        for (int k = 0; k < NE; k++) {
            const int e = lane + 64 * k;
            if (e < HD) hv[e] = hv[e] * r * in.wv[k];
        }
        wave_lds_sync();
    }
#pragma unroll
    for (int k = 0; k < NE; k++) {
        const int t = lane + 64 * k;
        if (t < half) {
            const float c = in.cs[k].x, sn = in.cs[k].y;
            const int ia = neox ? t : 2 * t, ib = neox ? t + half : 2 * t + 1;
            const float x0 = hv[ia], x1 = hv[ib];
            hv[ia] = x0 * c - x1 * sn;
            hv[ib] = x0 * sn + x1 * c;
        }
    }
    wave_lds_sync();
    EPI_TS(6);
}

// Decode (one row) scores with the q/k/v epilogue fused in: block = (kv head,
// chunk of ATT_CH positions), (gqa + 1) waves. Waves 0..gqa-1 post-process
// their query head; wave gqa post-processes the new k (and v) of the kv head
// and, in the block whose chunk holds the position, stores both into the
// cache. The chunk's K rows are staged in LDS (the new position's row from
// the post-processed k), then thread (query head, position) runs its dot
// product sequentially over the head dimension.
#ifndef QK_TS
#define QK_TS(i)
#endif
// (head_dim 256: at most 4 query heads per kv head, so that the block's
// 22 float4 of K per thread stay in registers)
constexpr int QKD_MAX_GQA_256 = 4;
template <int HD>
__global__ __launch_bounds__(HD == 256 ? 64 * (QKD_MAX_GQA_256 + 1) : 576) void k_attn_qk_decode(AttnArgs a, QkvPost p) {
    constexpr int KS = HD + 4;  // 16-byte rows; lanes reading 16 bytes of 16 rows hit all banks
    __shared__ __align__(16) float sk[ATT_CH * KS];
    __shared__ __align__(16) float sq[ATT_MAX_GQA + 1][HD];
    const int gqa = a.n_head / a.n_kv_head;
    const int lane = threadIdx.x & 63, hg = threadIdx.x >> 6;
    const int kvh = blockIdx.x, c = blockIdx.y;
    size_t t0, n;
    row_range(a, 0, t0, n);
    const size_t pos = n - 1;
    const size_t start = t0 + (size_t)c * ATT_CH;
    if (start >= n) return;
    const int rows = (int)min((size_t)ATT_CH, n - start);
    const size_t kv = (size_t)a.n_kv_head * HD;
    const float *cs_row = p.cs + pos * p.rot_dim;
    QK_TS(0);
    // the epilogue's inputs first, then the chunk's K rows, which do not
    // depend on it: the first PK float4 of each thread are in flight during
    // the epilogue (the new position's row is filled from the post-processed
    // k below)
    HeadIn<HD> hin;
    if (hg < gqa) {
        const int h = kvh * gqa + hg;
        head_load<HD>(hin, p.q + (size_t)h * HD, p.bq ? p.bq + (size_t)h * HD : nullptr, p.q_norm, cs_row, (int)p.rot_dim);
    } else {
        head_load<HD>(hin, p.k + (size_t)kvh * HD, p.bk ? p.bk + (size_t)kvh * HD : nullptr, p.k_norm, cs_row,
                      (int)p.rot_dim);
    }
    const float *kb = a.k_cache + start * kv + (size_t)kvh * HD;
    constexpr int R4 = HD / 4;
    // every float4 of the chunk a thread loads is in flight at once: up to
    // ATT_CH * HD / 4 over (gqa + 1) * 64 >= 192 threads (gqa >= 2 for
    // HD 256; smaller groups take the loop below for the rest)
    constexpr int PK = HD == 256 ? 22 : 8;
    const int nthreads = (gqa + 1) * 64;
    float4 kpre[PK];
#pragma unroll
    for (int j = 0; j < PK; j++) {
        const int idx = threadIdx.x + j * nthreads;
        const int r = idx / R4, c4 = idx % R4;
        kpre[j] = idx < rows * R4 && start + r != pos ? *(const float4 *)(kb + (size_t)r * kv + 4 * c4)
                                                      : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
    // the new position's k and v go to the cache only after the block's
    // barriers (a block barrier waits for the block's outstanding stores)
    const bool owner = hg == gqa && pos >= start && pos < start + ATT_CH;
    float vnew[HD / 64];
    if (owner)
#pragma unroll
        for (int j = 0; j < HD / 64; j++) {
            const int e = lane + 64 * j;
            vnew[j] = p.v[(size_t)kvh * HD + e];
            if (p.bv) vnew[j] = vnew[j] + p.bv[(size_t)kvh * HD + e];
        }
    if (hg < gqa) {
        head_post_wave<HD>(sq[hg], sk + hg * HD, hin, p.bq != nullptr, p.q_norm != nullptr, (int)p.rot_dim, p.neox, p.eps);
    } else {
        float *kn = sq[ATT_MAX_GQA];
        head_post_wave<HD>(kn, sk + gqa * HD, hin, p.bk != nullptr, p.k_norm != nullptr, (int)p.rot_dim, p.neox, p.eps);
    }
    QK_TS(1);
    __syncthreads();  // the epilogue used sk for the squares of the norms
    // K rows of the chunk into LDS (the new position from the post-processed k)
#pragma unroll
    for (int j = 0; j < PK; j++) {
        const int idx = threadIdx.x + j * nthreads;
        if (idx < rows * R4) {
            const int r = idx / R4, c4 = idx % R4;
            *(float4 *)(sk + r * KS + 4 * c4) = kpre[j];
        }
    }
    for (int idx = threadIdx.x + PK * nthreads; idx < rows * R4; idx += nthreads) {
        const int r = idx / R4, c4 = idx % R4;
        float4 k4;
        if (start + r == pos) k4 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        else k4 = *(const float4 *)(kb + (size_t)r * kv + 4 * c4);
        *(float4 *)(sk + r * KS + 4 * c4) = k4;
    }
    __syncthreads();
    if (pos >= start && pos < start + ATT_CH) {  // the new row
        const int r = (int)(pos - start);
        for (int e = threadIdx.x; e < HD; e += nthreads) sk[r * KS + e] = sq[ATT_MAX_GQA][e];
        __syncthreads();
    }
    QK_TS(2);
    if (owner) {
        float *kc = p.k_cache + pos * kv + (size_t)kvh * HD;
        float *vc = p.v_cache + pos * kv + (size_t)kvh * HD;
#pragma unroll
        for (int j = 0; j < HD / 64; j++) {
            kc[lane + 64 * j] = sq[ATT_MAX_GQA][lane + 64 * j];
            vc[lane + 64 * j] = vnew[j];
        }
    }
    if (hg >= gqa || lane >= rows) return;
    const float4 *kr = (const float4 *)(sk + lane * KS);
    const float4 *qq = (const float4 *)sq[hg];
    float sc = 0.0f;
#pragma unroll 8
    for (int d4 = 0; d4 < HD / 4; d4++) {
        const float4 k4 = kr[d4], q4 = qq[d4];
        sc += q4.x * k4.x;
        sc += q4.y * k4.y;
        sc += q4.z * k4.z;
        sc += q4.w * k4.w;
    }
    a.prob[(size_t)(kvh * gqa + hg) * a.span + (start + lane - t0)] = sc * a.scale;
    QK_TS(3);
}

// Softmax and output of one row per (head, group of SV_DB dims): block of
// SEQ_T threads.
//   softmax (ops.rs:98-112): max, glibc-matched exp, the sequential sum (one
//   thread for short spans, the exact parallel replay for spans of
//   SV_SEQ_MIN..SEQ_MAX_N), multiply by 1/sum; the blocks of one head repeat
//   it identically;
//   output (ops.rs:209-215): chunks of CP positions: all threads form the
//   products p_t * v_t,d into LDS, dim-major (row of dim d: CP products and
//   4 pad floats), with the float4 V loads issued PD chunks ahead; then
//   thread d adds its row in position order (lds_chain_chunks384, which does
//   not stop between chunks) while the others form the next chunk. Sixteen dims per block put 8 blocks on every head
//   (256 for 32 heads); chunks of 384 positions halve the barriers per
//   position against 192.
#ifndef ATT_TS
#define ATT_TS(i)
#endif
#ifndef SV_TS
#define SV_TS(c, i)
#endif
constexpr int ATT_MAX_SPAN = (int)ATT_MAX_CTX;
constexpr int SV_DB = 16;         // dims per block
constexpr int SV_CP = 384;        // positions per chunk
constexpr int SV_RS = SV_CP + 4;  // floats per dim row of the product buffer
constexpr int SV_BUF = SV_DB * SV_RS;  // floats per product buffer
constexpr int SV_SEQ_MIN = 1024;  // shorter spans are summed by one thread
template <int HD>
__global__ __launch_bounds__(SEQ_T) void k_attn_sv(AttnArgs a) {
    constexpr int DB = SV_DB;
    constexpr int CP = SV_CP;
    __shared__ __align__(16) float e[SEQ_PAD_N > ATT_MAX_SPAN + 64 ? SEQ_PAD_N : ATT_MAX_SPAN + 64];
    // product buffers / sum scratch
    __shared__ __align__(16) uint8_t ubuf[sizeof(SeqScratch) > 2 * SV_BUF * 4 ? sizeof(SeqScratch) : 2 * SV_BUF * 4];
    __shared__ float red[SEQ_T / 64];
    __shared__ float bc;
    __shared__ uint64_t stab[32];  // expf's 2^(i/32) table
    SeqScratch &S = *reinterpret_cast<SeqScratch *>(ubuf);
    float *prod = reinterpret_cast<float *>(ubuf);
    const int tid = threadIdx.x, lane = tid & 63;
    const int h = blockIdx.x / (HD / DB), d0 = (blockIdx.x % (HD / DB)) * DB;
    const int gqa = a.n_head / a.n_kv_head;
    const int kvh = h / gqa;
    size_t t0, n;
    row_range(a, 0, t0, n);
    const int cnt = (int)(n - t0);
    const bool exact = cnt >= SV_SEQ_MIN && cnt <= SEQ_MAX_N;
    const int C = seq_chunk(cnt);
    auto at = [&](int t) { return exact ? seq_idx(t, C) : t; };
    const float *ps = a.prob + (size_t)h * a.span;
    const size_t kv = (size_t)a.n_kv_head * HD;
    const float *vb = a.v_cache + t0 * kv + (size_t)kvh * HD + d0;
    constexpr int R4 = DB / 4;
    // wave 0 adds the products; the waves that do not share its SIMD (waves
    // are dealt to the 4 SIMDs in turn) form them, so the dependent adds
    // issue back to back
    constexpr int NPROD = (SEQ_T / 64 - SEQ_T / 256) * 64;
    static_assert(CP == 384, "the output adds run in lds_chain_chunks384");
    static_assert(CP * R4 == 2 * NPROD, "two float4 per producer thread per chunk");
    // V loads run PD chunks ahead of the products (a register ring)
    constexpr int PD = 8;
    float4 ring[PD][2];
    const int wv = tid >> 6;
    const int pid = (wv & 3) ? (wv - (wv >> 2) - 1) * 64 + lane : -1;
    auto issue = [&](float4 (&dst)[2], int c) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int idx = pid + k * NPROD;
            const int t = c * CP + idx / R4;
            dst[k] = t < cnt ? *(const float4 *)(vb + (size_t)t * kv + 4 * (idx % R4)) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
    };
    // the first PE chunks' V loads are in flight through the softmax (more
    // would hold registers the exact sum needs), the rest of the ring after it
    constexpr int PE = 2;
    if (pid >= 0)
#pragma unroll
        for (int j = 0; j < PE; j++) issue(ring[j], j);
    ATT_TS(0);
    // the scores stay in registers (all loads in flight together) through
    // the max; the exps, independent of each other, interleave
    constexpr int SPT = ATT_MAX_SPAN / SEQ_T;  // scores per thread
    exp_table_to_lds(stab);
    float sv[SPT];
    float mx = -INFINITY;
#pragma unroll
    for (int k = 0; k < SPT; k++) {
        const int t = tid + k * SEQ_T;
        sv[k] = t < cnt ? ps[t] : -INFINITY;
    }
#pragma unroll
    for (int k = 0; k < SPT; k++) mx = fmaxf(mx, sv[k]);
    mx = wave_max(mx);
    if (lane == 0) red[tid >> 6] = mx;
    __syncthreads();
    mx = wave_max(lane < SEQ_T / 64 ? red[lane] : -INFINITY);
    ATT_TS(1);
#pragma unroll
    for (int k = 0; k < SPT; k++) {
        const int t = tid + k * SEQ_T;
        if (t < cnt) e[at(t)] = aotk_expf_tab(sv[k] - mx, stab);
    }
    // the one-thread sum runs over whole runs of 64: the positions past the
    // span up to the next multiple of 64 hold -0.0, which leaves it unchanged
    if (!exact && tid < 64 && cnt + tid < ((cnt + 63) & ~63)) e[cnt + tid] = -0.0f;
    __syncthreads();
    ATT_TS(2);
    float sum;
    if (exact) {
        sum = exact_seq_sum(e, cnt, S);
    } else {
        if (tid == 0) bc = seq_sum_lds_pad64(e, cnt);
        __syncthreads();
        sum = bc;
    }
    const float inv = 1.0f / sum;
    for (int t = tid; t < cnt; t += SEQ_T) e[at(t)] = e[at(t)] * inv;
    __syncthreads();  // the sum's scratch is reused for the products below
    ATT_TS(3);
    float o = 0.0f;
    const int nch = (cnt + CP - 1) / CP;
    if (pid >= 0)
#pragma unroll
        for (int j = PE; j < PD; j++) issue(ring[j], j);
    // (a wave either adds or forms products; both sides meet nch barriers)
    if (__builtin_amdgcn_readfirstlane(wv) == 0) {
        if (tid < DB) o = lds_chain_chunks384(prod + tid * SV_RS, prod + SV_BUF + tid * SV_RS, (cnt + 63) >> 6, 0.0f);
    } else {
        for (int c0 = 0; c0 < nch; c0 += PD) {
#pragma unroll
            for (int j = 0; j < PD; j++) {
                const int c = c0 + j;
                if (c < nch) {
                    float *buf = prod + (c & 1) * SV_BUF;
                    const int base = c * CP;
                    const int rows = min(CP, cnt - base);
                    if (pid >= 0) {
#pragma unroll
                        for (int k = 0; k < 2; k++) {
                            const int idx = pid + k * NPROD;
                            const int r = idx / R4, d = 4 * (idx % R4);
                            // rows past the span hold -0.0, which leaves any sum unchanged
                            const bool in = r < rows;
                            const float pt = in ? e[at(base + r)] : 0.0f;
                            const float4 v4 = ring[j][k];
                            buf[(d + 0) * SV_RS + r] = in ? pt * v4.x : -0.0f;
                            buf[(d + 1) * SV_RS + r] = in ? pt * v4.y : -0.0f;
                            buf[(d + 2) * SV_RS + r] = in ? pt * v4.z : -0.0f;
                            buf[(d + 3) * SV_RS + r] = in ? pt * v4.w : -0.0f;
                        }
                        issue(ring[j], c + PD);
                    }
                    SV_TS(c, 0);
                    __syncthreads();
                    SV_TS(c, 1);
                }
            }
        }
    }
    ATT_TS(4);
    if (tid < DB) a.out[(size_t)h * HD + d0 + tid] = o;
}

// Decode attention in one launch for spans of at most AD_MAX_SPAN positions (the
// scores of k_attn_qk_decode and the softmax and output of k_attn_sv): block
// = (head, SV_DB dims) as in k_attn_sv. Wave 0 post-processes the head's q,
// wave 1 the kv head's new k (k_attn_qk_decode's epilogue, the same
// arithmetic), wave 2 loads the new v row; thread t then forms the score of
// position t0 + t (the sequential dot product over the head dimension, the
// new position's k from LDS) straight into registers, and the rest is
// k_attn_sv's code. Every block of the kv head computes the same new k and
// v; the first block of the kv head's first query head stores them into the
// cache, and the products of the new position take v from LDS (its cache
// row is not written yet when other blocks read). One launch fewer per
// layer than the scores + softmax/output pair, for the price of each head's
// scores formed by its HD / SV_DB blocks, each thread reading its position's
// K row (uncoalesced, from L2). Measured against the pair on Llama-3-8B
// decode: 486 -> 504 tok/s at ~140 positions, 480 -> 488 at ~270, 474 ->
// 468 at ~400, 463 -> 430 at ~640; TinyLlama's 38 positions 1080 -> 1159.
// Hence spans of up to 320 positions.
constexpr int AD_MAX_SPAN = 320;
template <int HD>
__global__ __launch_bounds__(SEQ_T) void k_attn_decode1(AttnArgs a, QkvPost p) {
    constexpr int DB = SV_DB;
    constexpr int CP = SV_CP;
    // scores / exps, padded to a run of 64 (spans below SV_SEQ_MIN: the one-thread sum)
    static_assert(AD_MAX_SPAN < SV_SEQ_MIN && AD_MAX_SPAN <= SEQ_T, "one position per thread, the one-thread sum");
    __shared__ __align__(16) float e[AD_MAX_SPAN + 64];
    __shared__ __align__(16) float prod[SV_BUF];
    __shared__ float red[SEQ_T / 64];
    __shared__ float bc;
    __shared__ uint64_t stab[32];  // expf's 2^(i/32) table
    __shared__ __align__(16) float hq[HD], hk[HD], hv[HD];  // post-processed q, new k, new v
    __shared__ __align__(16) float htmp[2][HD];             // the epilogue's norm scratch
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = tid >> 6;
    const int h = blockIdx.x / (HD / DB), d0 = (blockIdx.x % (HD / DB)) * DB;
    const int gqa = a.n_head / a.n_kv_head;
    const int kvh = h / gqa;
    size_t t0, n;
    row_range(a, 0, t0, n);
    const size_t pos = n - 1;
    const int cnt = (int)(n - t0);
    auto at = [&](int t) { return t; };
    const size_t kv = (size_t)a.n_kv_head * HD;
    const float *vb = a.v_cache + t0 * kv + (size_t)kvh * HD + d0;
    const float *cs_row = p.cs + pos * p.rot_dim;
    // the epilogue's inputs (waves 0 and 1) and the new v row (wave 2)
    HeadIn<HD> hin;
    if (wv == 0)
        head_load<HD>(hin, p.q + (size_t)h * HD, p.bq ? p.bq + (size_t)h * HD : nullptr, p.q_norm, cs_row, (int)p.rot_dim);
    else if (wv == 1)
        head_load<HD>(hin, p.k + (size_t)kvh * HD, p.bk ? p.bk + (size_t)kvh * HD : nullptr, p.k_norm, cs_row,
                      (int)p.rot_dim);
    else if (wv == 2)
        for (int e2 = lane; e2 < HD; e2 += 64) {
            float v = p.v[(size_t)kvh * HD + e2];
            if (p.bv) v = v + p.bv[(size_t)kvh * HD + e2];
            hv[e2] = v;
        }
    constexpr int R4 = DB / 4;
    constexpr int NPROD = (SEQ_T / 64 - SEQ_T / 256) * 64;
    static_assert(CP * R4 == 2 * NPROD && AD_MAX_SPAN <= CP, "one chunk, two float4 per producer thread");
    const int pid = (wv & 3) ? (wv - (wv >> 2) - 1) * 64 + lane : -1;
    float4 vin[2];  // in flight through the softmax
    if (pid >= 0)
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int idx = pid + k * NPROD;
            const int t = idx / R4;
            vin[k] = t < cnt ? *(const float4 *)(vb + (size_t)t * kv + 4 * (idx % R4)) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
    exp_table_to_lds(stab);
    if (wv == 0) head_post_wave<HD>(hq, htmp[0], hin, p.bq != nullptr, p.q_norm != nullptr, (int)p.rot_dim, p.neox, p.eps);
    else if (wv == 1) head_post_wave<HD>(hk, htmp[1], hin, p.bk != nullptr, p.k_norm != nullptr, (int)p.rot_dim, p.neox, p.eps);
    __syncthreads();
    // the new position's k and v into the cache: one block per kv head
    if (blockIdx.x == (unsigned)(kvh * gqa * (HD / DB)) && wv == 1) {
        float *kc = p.k_cache + pos * kv + (size_t)kvh * HD;
        float *vc = p.v_cache + pos * kv + (size_t)kvh * HD;
        for (int e2 = lane; e2 < HD; e2 += 64) {
            kc[e2] = hk[e2];
            vc[e2] = hv[e2];
        }
    }
    // the scores: thread t, position t0 + t (k_attn_qk_decode's dot product)
    float sv0 = -INFINITY;
    if (tid < cnt) {
        const float4 *kr = t0 + tid == pos ? (const float4 *)hk : (const float4 *)(a.k_cache + (t0 + tid) * kv + (size_t)kvh * HD);
        const float4 *qq = (const float4 *)hq;
        float sc = 0.0f;
#pragma unroll 8
        for (int d4 = 0; d4 < HD / 4; d4++) {
            const float4 k4 = kr[d4], q4 = qq[d4];
            sc += q4.x * k4.x;
            sc += q4.y * k4.y;
            sc += q4.z * k4.z;
            sc += q4.w * k4.w;
        }
        sv0 = sc * a.scale;
    }
    float mx = wave_max(sv0);
    if (lane == 0) red[wv] = mx;
    __syncthreads();
    mx = wave_max(lane < SEQ_T / 64 ? red[lane] : -INFINITY);
    if (tid < cnt) e[at(tid)] = aotk_expf_tab(sv0 - mx, stab);
    if (tid < 64 && cnt + tid < ((cnt + 63) & ~63)) e[cnt + tid] = -0.0f;
    __syncthreads();
    if (tid == 0) bc = seq_sum_lds_pad64(e, cnt);
    __syncthreads();
    const float sum = bc;
    const float inv = 1.0f / sum;
    for (int t = tid; t < cnt; t += SEQ_T) e[at(t)] = e[at(t)] * inv;
    __syncthreads();  // the sum's scratch is reused for the products below
    if (pid >= 0) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const int idx = pid + k * NPROD;
            const int r = idx / R4, d = 4 * (idx % R4);
            const bool in = r < cnt;
            const float pt = in ? e[at(r)] : 0.0f;
            // the new position's v from LDS (its cache row may not be written yet)
            const float4 v4 = r == cnt - 1 ? *(const float4 *)(hv + d0 + d) : vin[k];
            prod[(d + 0) * SV_RS + r] = in ? pt * v4.x : -0.0f;
            prod[(d + 1) * SV_RS + r] = in ? pt * v4.y : -0.0f;
            prod[(d + 2) * SV_RS + r] = in ? pt * v4.z : -0.0f;
            prod[(d + 3) * SV_RS + r] = in ? pt * v4.w : -0.0f;
        }
    }
    __syncthreads();
    if (tid < DB) a.out[(size_t)h * HD + d0 + tid] = lds_chain(prod + tid * SV_RS, (cnt + 63) >> 6, 0.0f);
}

// Batched rows (prompt chunks), spans up to ATT_MAX_SPAN: the same softmax
// and output, with the serial chains spread over lanes instead of blocks:
// k_attn_softmax_rows_p / _x, then k_attn_out_rows.

// Prompt output: wave = (kv head, 64 dimensions, NI consecutive items of
// (token, query head of the group)), lane = dimension: the lane's NI sums run
// over the positions in order, products by att_prod16 (lane 4K + i holds item
// i's probability of position K of each 16), one add per (item, position) on
// the VALU. V and the probabilities come straight from memory, 64 positions
// ahead in registers; the waves of a block (consecutive items of one kv head
// and slice) share V's lines in the L1. A wave alone on its SIMD issues an
// instruction per 4.7 clocks, which bounds it: 16 products and 16 NI adds per
// 16 positions, kept apart (a change between matrix and vector f32 costs 14).
template <int HD, int NI>
__global__ __launch_bounds__(256, 1) void k_attn_out_rows(AttnArgs a, int m) {
    constexpr int NS = HD / 64;
    const int gqa = a.n_head / a.n_kv_head;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int slice = blockIdx.x % NS, kvh = (blockIdx.x / NS) % a.n_kv_head;
    const int items = m * gqa, it0 = (blockIdx.x / (NS * a.n_kv_head) * 4 + wave) * NI;
    if (it0 >= items) return;
    const size_t kv = (size_t)a.n_kv_head * HD;
    // the items' ranges (items past the last repeat it, unstored), from the first one's start
    size_t lo, tmp;
    row_range(a, (size_t)(it0 / gqa), lo, tmp);
    int t0[NI], tn[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) {
        size_t x, y;
        row_range(a, (size_t)(min(it0 + i, items - 1) / gqa), x, y);
        t0[i] = (int)(x - lo);
        tn[i] = (int)(y - lo);
    }
    const int alo = t0[NI - 1], ahi = tn[0], cnt = tn[NI - 1];  // common to all: [alo, ahi)
    // groups of 16 positions that all items hold: [gs, ge)
    const int gs = (alo + 15) >> 4, ge = max(gs, ahi >> 4);
    // this lane's probability operand: item lane % 4, position lane / 4 of each 16
    const int mine = min(it0 + min(lane & 3, NI - 1), items - 1), mt = mine / gqa;
    const float *pr = a.prob + ((size_t)mt * a.n_head + (size_t)kvh * gqa + mine % gqa) * a.span;
    size_t mx, my;
    row_range(a, (size_t)mt, mx, my);
    const int m0 = (int)(mx - lo), m1 = (int)(my - lo);
    const float *vb = a.v_cache + lo * kv + (size_t)kvh * HD + slice * 64;  // (wave-uniform)
    float o[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) o[i] = 0.0f;
    auto load_p = [&](int t) { return pr[max(min(t + (lane >> 2), m1 - 1), m0) - m0]; };
    // a group that some item does not hold whole, or past the end
    auto edge = [&](int g) {
        const int t = 16 * g;
        float y[16];
        att_f4 x[16];
#pragma unroll
        for (int k = 0; k < 16; k++) y[k] = vb[(size_t)min(t + k, cnt - 1) * kv + lane];
        att_prod16(x, load_p(t), y);
#pragma unroll
        for (int k = 0; k < 16; k++)
#pragma unroll
            for (int i = 0; i < NI; i++)
                if (t + k >= t0[i] && t + k < tn[i]) o[i] += x[k][i];
    };
    for (int g = 0; g < gs; g++) edge(g);
    if (gs < ge) {
        constexpr int PD = 4;  // groups in flight
        float v[PD][16], p[PD];
        uint32_t off[16];  // a group's rows from its first: one base per group, no address arithmetic per load
#pragma unroll
        for (int k = 0; k < 16; k++) off[k] = (uint32_t)((size_t)k * kv) + lane;
        auto load = [&](float (&vv)[16], float &pp, int g) {  // (groups past the last re-read it: never used)
            const int t = 16 * min(g, ge - 1);
            const float *base = vb + (size_t)t * kv;
#pragma unroll
            for (int k = 0; k < 16; k++) vv[k] = base[off[k]];
            pp = load_p(t);
        };
        auto add = [&](const att_f4 (&x)[16]) {
#pragma unroll
            for (int k = 0; k < 16; k++)
#pragma unroll
                for (int i = 0; i < NI; i++) o[i] += x[k][i];
#pragma unroll
            for (int i = 0; i < NI; i++) asm volatile("" : "+v"(o[i]));
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int k = 0; k < PD; k++) load(v[k], p[k], gs + k);
        __builtin_amdgcn_sched_barrier(0);
        // the products of a group are formed before the sums of the one before it
        att_f4 x0[16], x1[16];
        att_prod16(x0, p[0], v[0]);
        load(v[0], p[0], gs + PD);
        __builtin_amdgcn_sched_barrier(0);
        int g = gs;
        for (; g + PD <= ge; g += PD) {
#pragma unroll
            for (int k = 0; k < PD; k++) {
                att_prod16(k & 1 ? x0 : x1, p[(k + 1) % PD], v[(k + 1) % PD]);
                load(v[(k + 1) % PD], p[(k + 1) % PD], g + k + 1 + PD);
                __builtin_amdgcn_sched_barrier(0);
                add(k & 1 ? x1 : x0);
            }
        }
#pragma unroll
        for (int k = 0; k < PD - 1; k++) {
            if (g + k < ge) {
                att_prod16(k & 1 ? x0 : x1, p[(k + 1) % PD], v[(k + 1) % PD]);
                add(k & 1 ? x1 : x0);
            }
        }
    }
    for (int g = ge; 16 * g < cnt; g++) edge(g);
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int it = it0 + i;
        if (it < items) a.out[(size_t)(it / gqa) * a.n_head * HD + (size_t)(kvh * gqa + it % gqa) * HD + slice * 64 + lane] = o[i];
    }
}

// Softmax of few long rows: a block of SEQ_T threads per (row, head), the
// scores held in registers through the max, the exps with the 2^(i/32) table
// in LDS, the exact parallel replay of the sequential sum.
template <int CAP>
__global__ __launch_bounds__(SEQ_T) void k_attn_softmax_rows_x(AttnArgs a, int m) {
    __shared__ __align__(16) float e[CAP + SEQ_T + 32];
    __shared__ SeqScratch S;
    __shared__ float red[SEQ_T / 64];
    __shared__ uint64_t stab[32];
    constexpr int SPT = CAP / SEQ_T;
    const int tid = threadIdx.x, lane = tid & 63;
    const int i = blockIdx.x / a.n_head, h = blockIdx.x % a.n_head;
    size_t t0, n;
    row_range(a, i, t0, n);
    const int cnt = (int)(n - t0);
    float *ps = a.prob + ((size_t)i * a.n_head + h) * a.span;
    exp_table_to_lds(stab);
    float sv[SPT];
    float mx = -INFINITY;
#pragma unroll
    for (int k = 0; k < SPT; k++) {
        const int t = tid + k * SEQ_T;
        sv[k] = t < cnt ? ps[t] : -INFINITY;
        mx = fmaxf(mx, sv[k]);
    }
    mx = wave_max(mx);
    if (lane == 0) red[tid >> 6] = mx;
    __syncthreads();
    mx = wave_max(lane < SEQ_T / 64 ? red[lane] : -INFINITY);
    const int C = seq_chunk(cnt);
#pragma unroll
    for (int k = 0; k < SPT; k++) {
        const int t = tid + k * SEQ_T;
        if (t < cnt) {
            sv[k] = aotk_expf_tab(sv[k] - mx, stab);
            e[seq_idx(t, C)] = sv[k];
        }
    }
    __syncthreads();
    const float inv = 1.0f / exact_seq_sum(e, cnt, S);
#pragma unroll
    for (int k = 0; k < SPT; k++) {
        const int t = tid + k * SEQ_T;
        if (t < cnt) ps[t] = sv[k] * inv;
    }
}

// Softmax of prompt rows: P (row, head) pairs per block of T threads, each on
// T / P of them with its scores in registers: max, glibc-matched exp into
// LDS, the P sequential sums side by side, one per lane of wave 0 (rows 16
// bytes apart in the banks), then p = e * (1 / sum) over the scores. The
// chain's latency (about 7 clocks per position) bounds it: paid once per
// block, and hidden by the loads and exps of other blocks only where several
// fit a CU.
template <int P, int CAP, int T>
__global__ __launch_bounds__(T) void k_attn_softmax_rows_p(AttnArgs a, int m) {
    constexpr int TP = T / P, NV = CAP / TP / 4, NW = TP / 64, RS = CAP + 4;
    __shared__ __align__(16) float e[P * RS];
    __shared__ float red[T / 64], sinv[P];
    __shared__ uint64_t stab[32];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int r = tid / TP, u = tid % TP;
    const int pairs = m * a.n_head, pair = min((int)blockIdx.x * P + r, pairs - 1);  // pairs past the last repeat it, unstored
    const bool own = (int)blockIdx.x * P + r < pairs;
    size_t t0, n, n_last;
    row_range(a, (size_t)(pair / a.n_head), t0, n);
    const int cnt = (int)(n - t0);
    // the block's longest row, in whole runs of 64 (ranges grow with the row)
    row_range(a, (size_t)(min((int)blockIdx.x * P + P - 1, pairs - 1) / a.n_head), t0, n_last);
    const int run = ((int)(n_last - t0) + 63) & ~63;
    float4 *ps = (float4 *)(a.prob + (size_t)pair * a.span);
    exp_table_to_lds(stab);
    float4 v[NV];
    float mx = -INFINITY;
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const int t = 4 * (u + TP * k);
        v[k] = t < cnt ? ps[u + TP * k] : make_float4(-INFINITY, -INFINITY, -INFINITY, -INFINITY);  // (rows are whole float4s)
        if (t + 1 >= cnt) v[k].y = -INFINITY;
        if (t + 2 >= cnt) v[k].z = -INFINITY;
        if (t + 3 >= cnt) v[k].w = -INFINITY;
    }
#pragma unroll
    for (int k = 0; k < NV; k++) mx = fmaxf(mx, fmaxf(fmaxf(v[k].x, v[k].y), fmaxf(v[k].z, v[k].w)));
    mx = wave_max(mx);
    if (lane == 0) red[w] = mx;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NW; k++) mx = fmaxf(mx, red[r * NW + k]);
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const int t = 4 * (u + TP * k);
        if (t < run) {
            // -0 past the row's end: neutral in the sum
            v[k].x = t < cnt ? aotk_expf_tab(v[k].x - mx, stab) : -0.0f;
            v[k].y = t + 1 < cnt ? aotk_expf_tab(v[k].y - mx, stab) : -0.0f;
            v[k].z = t + 2 < cnt ? aotk_expf_tab(v[k].z - mx, stab) : -0.0f;
            v[k].w = t + 3 < cnt ? aotk_expf_tab(v[k].w - mx, stab) : -0.0f;
            *(float4 *)&e[r * RS + t] = v[k];
        }
    }
    __syncthreads();
    if (tid < P) sinv[tid] = 1.0f / seq_sum_lds_pad64(e + tid * RS, run);
    __syncthreads();
    const float inv = sinv[r];
    if (!own) return;
#pragma unroll
    for (int k = 0; k < NV; k++) {
        const int t = 4 * (u + TP * k);
        if (t < cnt) ps[u + TP * k] = make_float4(v[k].x * inv, v[k].y * inv, v[k].z * inv, v[k].w * inv);
    }
}

static void launch_rows(const AttnArgs &a, size_t head_dim, size_t m, size_t longest, hipStream_t s) {
    const unsigned pairs = (unsigned)(m * a.n_head);
#define SML(P, CAP, T) k_attn_softmax_rows_p<P, CAP, T><<<(pairs + P - 1) / P, T, 0, s>>>(a, (int)m)
    if (pairs >= 1024 && longest <= 8192) {
        // enough pairs for eight per block on every CU (four past 4096
        // positions: LDS). 64 rows x 32 heads, against one pair per wave and,
        // past 1024 positions, 256 threads with the parallel replay: 500
        // positions 10.0 -> 6.2 us, 1000 16.5 -> 9.9, 2000 31 -> 16.5, 4090 49
        // -> 31, 6064 95 -> 65, 8100 112 -> 83. Against the replay of _x there:
        // 34, 38, 45, 54, 66, 75; at 1024 pairs 2000 positions 15.6 / 23.5 us,
        // 4090 27.8 / 28.5, 8100 44 / 41; at 768 pairs 3000 21.3 / 20.0, 4090
        // 27.2 / 22.0. The next larger instance costs 0.1..0.9 us: 500
        // positions 6.3, 1000 10.2, 2000 16.7.
        if (longest <= 512) SML(8, 512, 1024);
        else if (longest <= 1024) SML(8, 1024, 1024);
        else if (longest <= 2048) SML(8, 2048, 1024);
        else if (longest <= 4096) SML(8, 4096, 1024);
        else SML(4, 8192, 1024);
    } else if (longest <= 2048) {
        // few pairs: more threads each. Against one pair per wave before: 50
        // rows x 8 heads, a 1024 window 17.7 -> 6.5 us; 6 rows x 32 heads, 2006
        // positions 34 -> 11.4. Against eight per block, 512 pairs: 500
        // positions 5.6 / 6.0, 1000 7.4 / 9.2, 2000 12.0 / 15.6. (Measured, not
        // used: at 64..256 pairs the replay is ahead from 1000 positions on,
        // 2000 in 7.2 us; at 768 pairs eight per block from 1500, 2000 in 15.7
        // against 19.3.)
        if (longest <= 512) SML(4, 512, 512);
        else if (longest <= 1024) SML(2, 1024, 512);
        else SML(2, 2048, 1024);
    } else if (longest <= 8192) {
        // few long rows: the parallel replay (20 rows x 8 heads, 3020
        // positions: 7.0 us against 18 for four per block; 512 pairs, 4090
        // positions 15.5 / 23)
        k_attn_softmax_rows_x<8192><<<pairs, SEQ_T, 0, s>>>(a, (int)m);
    } else {
        k_attn_softmax_rows_x<ATT_MAX_SPAN><<<pairs, SEQ_T, 0, s>>>(a, (int)m);
    }
#undef SML
    // Items per wave: as many waves as there are SIMDs first, then more items
    // per product (each product instruction serves up to four). 64 rows x 32
    // heads x 4032 positions (4096 / NI waves): NI 4 79..88 us over a run, 2
    // 115, 1 205 (117 before, with V per wave from L2 and p from LDS); 64 rows
    // x 8 heads x 7000, head_dim 256: NI 2 118, 4 133, 1 176 (159); 6 rows x 32
    // heads x 2000: NI 1 29, 2 35, 4 41 (45).
    const size_t items = m * (a.n_head / a.n_kv_head), per = a.n_kv_head * (head_dim / 64);
    const int NI = items * per <= 1024 ? 1 : items * per <= 2048 ? 2 : 4;
    const unsigned g = (unsigned)(per * ((items + 4 * NI - 1) / (4 * NI)));
#define OUTL(H)                                                              \
    do {                                                                     \
        if (NI == 1) k_attn_out_rows<H, 1><<<g, 256, 0, s>>>(a, (int)m);     \
        else if (NI == 2) k_attn_out_rows<H, 2><<<g, 256, 0, s>>>(a, (int)m); \
        else k_attn_out_rows<H, 4><<<g, 256, 0, s>>>(a, (int)m);             \
    } while (0)
    if (head_dim == 64) OUTL(64);
    else if (head_dim == 128) OUTL(128);
    else OUTL(256);
#undef OUTL
}

static void launch_sv(const AttnArgs &a, size_t head_dim, hipStream_t s) {
    const unsigned g = (unsigned)(a.n_head * (head_dim / SV_DB));
    switch (head_dim) {
    case 64: k_attn_sv<64><<<g, SEQ_T, 0, s>>>(a); break;
    case 128: k_attn_sv<128><<<g, SEQ_T, 0, s>>>(a); break;
    default: k_attn_sv<256><<<g, SEQ_T, 0, s>>>(a); break;
    }
}

size_t attention_scratch_bytes(size_t n_head, size_t head_dim, size_t ctx, size_t m) {
    (void)head_dim;
    return align_up(m * n_head * align_up(ctx, 4) * 4, 256);
}

static AttnArgs attn_args(float *out, const float *q, const float *k_cache, const float *v_cache, size_t n_head,
                          size_t n_kv_head, size_t head_dim, size_t ctx_rows, size_t pos0, size_t window,
                          const int *pos_dev, float *scratch) {
    AttnArgs a;
    a.out = out;
    a.q = q;
    a.k_cache = k_cache;
    a.v_cache = v_cache;
    a.prob = scratch;
    a.span = (int)align_up(ctx_rows, 4);
    a.n_head = (int)n_head;
    a.n_kv_head = (int)n_kv_head;
    a.hd = (int)head_dim;
    a.pos0 = pos0;
    a.window = window;
    a.pos_dev = pos_dev;
    a.scale = 1.0f / sqrtf((float)head_dim);
    return a;
}

void launch_attention(float *out, const float *q, const float *k_cache, const float *v_cache, size_t n_head,
                      size_t n_kv_head, size_t head_dim, size_t ctx_rows, size_t pos0, size_t m, size_t window,
                      float *scratch, hipStream_t s) {
    AttnArgs a = attn_args(out, q, k_cache, v_cache, n_head, n_kv_head, head_dim, ctx_rows, pos0, window, nullptr,
                           scratch);
    if (m > 1) {
        // Eight rows per wave where that still leaves about four blocks per
        // CU, else four. 64 rows: 32 heads x 4032 positions, head_dim 128,
        // 59..66 us over a run with eight, 69 with four (102 before); 8 heads x
        // 7000, head_dim 256, 57 / 64 (147); 32 heads x 448 14.7 / 14.2 (17.6);
        // 8 heads, a 1024 window, head_dim 256, 21.4 / 20.1 (40); 6 rows x 32
        // heads x 2000 9.6 / 8.5 (10.6).
        const size_t held = window > 0 && window < pos0 + m ? window + m : pos0 + m;  // positions of any row
        const int gqa = (int)(n_head / n_kv_head), rgs = std::max(1, 4 / gqa);
        const size_t blocks8 = n_kv_head * ((held + ATT_CH - 1) / ATT_CH) * ((m + 8 * rgs - 1) / (8 * rgs));
        const int R = blocks8 >= 1024 ? 8 : 4;
        const dim3 g((unsigned)n_kv_head, (unsigned)((pos0 + m + ATT_CH - 1) / ATT_CH), (unsigned)((m + R * rgs - 1) / (R * rgs)));
        const unsigned th = (unsigned)(64 * gqa * rgs);
#define SCL(H)                                                              \
    do {                                                                    \
        if (R == 4) k_attn_scores_rows<H, 1><<<g, th, 0, s>>>(a, (int)m, rgs); \
        else k_attn_scores_rows<H, 2><<<g, th, 0, s>>>(a, (int)m, rgs);      \
    } while (0)
        if (head_dim == 64) SCL(64);
        else if (head_dim == 128) SCL(128);
        else SCL(256);
#undef SCL
        // the longest row spans min(pos0 + m, window) positions
        launch_rows(a, head_dim, m, window > 0 && window < pos0 + m ? window : pos0 + m, s);
        return;
    }
    const size_t span = window > 0 && window < ctx_rows ? window : ctx_rows;
    const dim3 grid((unsigned)n_kv_head, (unsigned)((span + ATT_CH - 1) / ATT_CH));
    const unsigned threads = (unsigned)(64 * (n_head / n_kv_head));
    switch (head_dim) {
    case 64: k_attn_scores<64><<<grid, threads, 0, s>>>(a); break;
    case 128: k_attn_scores<128><<<grid, threads, 0, s>>>(a); break;
    default: k_attn_scores<256><<<grid, threads, 0, s>>>(a); break;
    }
    launch_sv(a, head_dim, s);
}

void launch_attention_decode(float *out, const QkvPost &p, size_t ctx_rows, size_t pos0, size_t window,
                             const int *pos_dev, float *scratch, hipStream_t s) {
    AttnArgs a = attn_args(out, p.q, p.k_cache, p.v_cache, p.n_head, p.n_kv_head, p.head_dim, ctx_rows, pos0, window,
                           pos_dev, scratch);
    size_t span = window > 0 && window < ctx_rows ? window : ctx_rows;
    if (span <= (size_t)AD_MAX_SPAN) {  // short spans: scores, softmax and output in one launch
        const dim3 g1((unsigned)(p.n_head * (p.head_dim / SV_DB)), 1);
        switch (p.head_dim) {
        case 64: k_attn_decode1<64><<<g1, SEQ_T, 0, s>>>(a, p); break;
        case 128: k_attn_decode1<128><<<g1, SEQ_T, 0, s>>>(a, p); break;
        default: k_attn_decode1<256><<<g1, SEQ_T, 0, s>>>(a, p); break;
        }
        return;
    }
    dim3 grid((unsigned)p.n_kv_head, (unsigned)((span + ATT_CH - 1) / ATT_CH), 1);
    const unsigned threads = (unsigned)(64 * (p.n_head / p.n_kv_head + 1));
    switch (p.head_dim) {
    case 64: k_attn_qk_decode<64><<<grid, threads, 0, s>>>(a, p); break;
    case 128: k_attn_qk_decode<128><<<grid, threads, 0, s>>>(a, p); break;
    default: k_attn_qk_decode<256><<<grid, threads, 0, s>>>(a, p); break;
    }
    launch_sv(a, p.head_dim, s);
}

// ------------------------------------------------------------ elementwise

__global__ void k_add(float *x, const float *y, size_t n) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) x[i] = x[i] + y[i];
}
void launch_add(float *x, const float *y, size_t n, hipStream_t s) {
    k_add<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(x, y, n);
}

// Gemma post-norm join: x += rmsnorm(y) (emit.rs:320-324).
__global__ __launch_bounds__(SEQ_T) void k_rmsnorm_add(float *x, const float *y, const float *w, int n, float eps) {
    __shared__ float sq[SEQ_PAD_N];
    __shared__ SeqScratch S;
    const size_t m = blockIdx.x;
    const float *yr = y + m * n;
    float *xr = x + m * n;
    const int C = seq_chunk(n);
    // every load (y, and x and w for the update) is issued before the sum, y
    // first: the loads complete in order, so the squares wait for y only
    float yv[8], xv[8], wv[8];
#pragma unroll
    for (int k = 0; k < 8; k++) yv[k] = yr[min((int)threadIdx.x + k * SEQ_T, n - 1)];
#pragma unroll
    for (int k = 0; k < 8; k++) xv[k] = xr[min((int)threadIdx.x + k * SEQ_T, n - 1)];
#pragma unroll
    for (int k = 0; k < 8; k++) wv[k] = w[min((int)threadIdx.x + k * SEQ_T, n - 1)];
    // y is needed here, on every path: no load may move into the conditional
    // stores below (and wait there for x and w)
#pragma unroll
    for (int k = 0; k < 8; k++) asm volatile("" : "+v"(yv[k]));
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int i = threadIdx.x + k * SEQ_T;
        if (i < n) sq[seq_idx(i, C)] = yv[k] * yv[k];
    }
    __syncthreads();
    RMS_TS(1);
    float ss = exact_seq_sum(sq, n, S);
    RMS_TS(2);
    float r = 1.0f / sqrtf(ss / (float)n + eps);
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int i = threadIdx.x + k * SEQ_T;
        if (i < n) xr[i] = xv[k] + yv[k] * r * wv[k];
    }
}
// Gemma: the post-norm join x += rmsnorm(y) (emit.rs:320-324) and the next
// rmsnorm of x with its quantization (the following block's input), in one
// launch: the updated row stays in registers between the two exact sums.
__global__ __launch_bounds__(SEQ_T) void k_rmsnorm_add_quant(float *x, const float *y, const float *w_post,
                                                             const float *w_next, int n, float eps, RmsOut out) {
    __shared__ __align__(16) float row[8192];
    __shared__ float sq[SEQ_PAD_N];
    __shared__ SeqScratch S;
    const size_t m = blockIdx.x;
    const float *yr = y + m * n;
    float *xr = x + m * n;
    const int C = seq_chunk(n);
    float yv[8], xv[8], wv[8], wn[8];
#pragma unroll
    for (int k = 0; k < 8; k++) yv[k] = yr[min((int)threadIdx.x + k * SEQ_T, n - 1)];
#pragma unroll
    for (int k = 0; k < 8; k++) xv[k] = xr[min((int)threadIdx.x + k * SEQ_T, n - 1)];
#pragma unroll
    for (int k = 0; k < 8; k++) wv[k] = w_post[min((int)threadIdx.x + k * SEQ_T, n - 1)];
#pragma unroll
    for (int k = 0; k < 8; k++) wn[k] = w_next[min((int)threadIdx.x + k * SEQ_T, n - 1)];
#pragma unroll
    for (int k = 0; k < 8; k++) asm volatile("" : "+v"(yv[k]));
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int i = threadIdx.x + k * SEQ_T;
        if (i < n) sq[seq_idx(i, C)] = yv[k] * yv[k];
    }
    __syncthreads();
    const float ss = exact_seq_sum(sq, n, S);
    const float r = 1.0f / sqrtf(ss / (float)n + eps);
    // x += y * r * w (as k_rmsnorm_add), then the squares of the new x
    // (exact_seq_sum's closing barrier orders these writes after its reads)
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int i = threadIdx.x + k * SEQ_T;
        if (i < n) {
            const float v = xv[k] + yv[k] * r * wv[k];
            xv[k] = v;
            row[i] = v;
            sq[seq_idx(i, C)] = v * v;
        }
    }
    __syncthreads();
    const float ss2 = exact_seq_sum(sq, n, S);
    const float r2 = 1.0f / sqrtf(ss2 / (float)n + eps);
#pragma unroll
    for (int k = 0; k < 8; k++) {
        const int i = threadIdx.x + k * SEQ_T;
        if (i < n) {
            xr[i] = xv[k];  // stored after the sums (see k_rmsnorm_add_quant4)
            const float v = row[i] * r2 * wn[k];
            row[i] = v;
            if (out.f32) out.f32[m * n + i] = v;
        }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    ActQ8K qk = q8k_row(out.q8k, m, n);
    ActQ8_0 q0 = q80_row(out.q80, m, n);
    for (int b = wave; b < n / 256; b += nw) {
        float4 v4 = ((const float4 *)(row + b * 256))[lane];
        float v[4] = {v4.x, v4.y, v4.z, v4.w};
        quant256(v, lane, b, qk, q0);
    }
}

// The same for rows of whole 256-blocks, float4 per thread as in
// k_rmsnorm_quant4 (the joined row quantized from registers).
template <int KF>
__global__ __launch_bounds__(SEQ_T) void k_rmsnorm_add_quant4(float *x, const float *y, const float *w_post,
                                                              const float *w_next, int n, float eps, RmsOut out) {
    __shared__ float sq[SEQ_PAD_N];
    __shared__ SeqScratch S;
    const size_t m = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63;
    const int n4 = n / 4;
    const int C = seq_chunk(n);
    float4 *xr = (float4 *)(x + m * n);
    const float4 *yr = (const float4 *)(y + m * n);
    float4 yv[KF], xv[KF], wv[KF], wn[KF];
    const float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
#pragma unroll
    for (int k = 0; k < KF; k++) yv[k] = tid + k * SEQ_T < n4 ? yr[tid + k * SEQ_T] : z;
#pragma unroll
    for (int k = 0; k < KF; k++) xv[k] = tid + k * SEQ_T < n4 ? xr[tid + k * SEQ_T] : z;
#pragma unroll
    for (int k = 0; k < KF; k++) wv[k] = tid + k * SEQ_T < n4 ? ((const float4 *)w_post)[tid + k * SEQ_T] : z;
#pragma unroll
    for (int k = 0; k < KF; k++) wn[k] = tid + k * SEQ_T < n4 ? ((const float4 *)w_next)[tid + k * SEQ_T] : z;
    auto squares = [&](const float4 &v, int i) {
        sq[seq_idx(4 * i, C)] = v.x * v.x;
        sq[seq_idx(4 * i + 1, C)] = v.y * v.y;
        sq[seq_idx(4 * i + 2, C)] = v.z * v.z;
        sq[seq_idx(4 * i + 3, C)] = v.w * v.w;
    };
#pragma unroll
    for (int k = 0; k < KF; k++)
        if (tid + k * SEQ_T < n4) squares(yv[k], tid + k * SEQ_T);
    __syncthreads();
    const float ss = exact_seq_sum(sq, n, S);
    const float r = 1.0f / sqrtf(ss / (float)n + eps);
    // x += y * r * w (as k_rmsnorm_add), then the squares of the new x
    // (exact_seq_sum's closing barrier orders these writes after its reads)
#pragma unroll
    for (int k = 0; k < KF; k++) {
        const int i = tid + k * SEQ_T;
        if (i < n4) {
            float4 v;
            v.x = xv[k].x + yv[k].x * r * wv[k].x;
            v.y = xv[k].y + yv[k].y * r * wv[k].y;
            v.z = xv[k].z + yv[k].z * r * wv[k].z;
            v.w = xv[k].w + yv[k].w * r * wv[k].w;
            xv[k] = v;
            squares(v, i);
        }
    }
    __syncthreads();
    const float ss2 = exact_seq_sum(sq, n, S);
    const float r2 = 1.0f / sqrtf(ss2 / (float)n + eps);
    const ActQ8K qk = q8k_row(out.q8k, m, n);
    const ActQ8_0 q0 = q80_row(out.q80, m, n);
    // the new x is stored only now: a store in flight would hold up every
    // barrier of the second sum (a block barrier waits for the block's
    // outstanding memory operations)
#pragma unroll
    for (int k = 0; k < KF; k++) {
        const int i = tid + k * SEQ_T;
        if (i < n4) xr[i] = xv[k];
    }
#pragma unroll
    for (int k = 0; k < KF; k++) {
        const int i = tid + k * SEQ_T;
        if (i < n4) {  // wave-uniform: n4 is a multiple of 64
            const float v[4] = {xv[k].x * r2 * wn[k].x, xv[k].y * r2 * wn[k].y, xv[k].z * r2 * wn[k].z, xv[k].w * r2 * wn[k].w};
            if (out.f32) *(float4 *)(out.f32 + m * n + 4 * i) = make_float4(v[0], v[1], v[2], v[3]);
            quant256(v, lane, (size_t)(i >> 6), qk, q0);
        }
    }
}

void launch_rmsnorm_add_quant(float *x, const float *y, const float *w_post, const float *w_next, size_t n, size_t m,
                              float eps, RmsOut out, hipStream_t s) {
    if (m < 2) out.q8k.qt = nullptr, out.q80.xh = nullptr;  // the tiled / f16 copies serve batches only
    if (n % 256 == 0 && n <= 4096) k_rmsnorm_add_quant4<1><<<(unsigned)m, SEQ_T, 0, s>>>(x, y, w_post, w_next, (int)n, eps, out);
    else if (n % 256 == 0) k_rmsnorm_add_quant4<2><<<(unsigned)m, SEQ_T, 0, s>>>(x, y, w_post, w_next, (int)n, eps, out);
    else k_rmsnorm_add_quant<<<(unsigned)m, SEQ_T, 0, s>>>(x, y, w_post, w_next, (int)n, eps, out);
}

void launch_rmsnorm_add(float *x, const float *y, const float *w, size_t n, size_t m, float eps, hipStream_t s) {
    k_rmsnorm_add<<<(unsigned)m, SEQ_T, 0, s>>>(x, y, w, (int)n, eps);
}

__global__ void k_silu_mul(float *h, const float *up, size_t n, int gelu) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    h[i] = gelu ? gelu_f(h[i]) * up[i] : silu_f(h[i], up[i]);
}
void launch_silu_mul(float *h, const float *up, size_t n, int gelu, hipStream_t s) {
    k_silu_mul<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(h, up, n, gelu);
}

// softmax (ops.rs:98-112) of one vector: max, exp, sequential sum, scale.
__global__ __launch_bounds__(SEQ_T) void k_softmax(float *x, int n) {
    __shared__ float red[16];
    __shared__ float bc;
    __shared__ float ev[SEQ_PAD_N];
    __shared__ SeqScratch S;
    float mx = -INFINITY;
    for (int i = threadIdx.x; i < n; i += blockDim.x) mx = fmaxf(mx, x[i]);
    mx = wave_max(mx);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = mx;
    __syncthreads();
    float t = (threadIdx.x & 63) < (blockDim.x >> 6) ? red[threadIdx.x & 63] : -INFINITY;
    mx = wave_max(t);
    for (int i = threadIdx.x; i < n; i += blockDim.x) x[i] = aotk_expf(x[i] - mx);
    __syncthreads();
    float sum;
    if (n <= SEQ_MAX_N) {
        const int C = seq_chunk(n);
        for (int i = threadIdx.x; i < n; i += blockDim.x) ev[seq_idx(i, C)] = x[i];
        __syncthreads();
        sum = exact_seq_sum(ev, n, S);
    } else {
        if (threadIdx.x == 0) {
            float t = 0.0f;
            for (int i = 0; i < n; i++) t += x[i];
            bc = t;
        }
        __syncthreads();
        sum = bc;
    }
    float inv = 1.0f / sum;
    for (int i = threadIdx.x; i < n; i += blockDim.x) x[i] = x[i] * inv;
}
void launch_softmax(float *x, size_t n, hipStream_t s) { k_softmax<<<1, SEQ_T, 0, s>>>(x, (int)n); }

void launch_rmsnorm_heads(float *x, const float *w, size_t n_heads, size_t head_dim, float eps, hipStream_t s) {
    QkvPost p = {};
    p.q = x;
    p.q_norm = w;
    p.n_head = n_heads;
    p.n_kv_head = 0;
    p.head_dim = head_dim;
    p.rot_dim = 0;
    p.eps = eps;
    static float dummy_cs[2];
    (void)dummy_cs;
    p.cs = x;  // unused with rot_dim == 0
    launch_qkv_post(p, 1, 0, nullptr, s);
}

void launch_rope(float *x, size_t m, size_t n_heads, size_t head_dim, size_t rot_dim, const float *cs, int neox,
                 hipStream_t s) {
    // positions 0..m-1 index the m rows of the table
    QkvPost p = {};
    p.q = x;
    p.n_head = n_heads;
    p.n_kv_head = 0;
    p.head_dim = head_dim;
    p.rot_dim = rot_dim;
    p.cs = cs;
    p.neox = neox;
    launch_qkv_post(p, m, 0, nullptr, s);
}

// ----------------------------------------------------------------- argmax
// First index of the strict maximum (sampler.rs:99-109): -inf and NaN never
// win; an empty / all -inf input gives 0.
__device__ __forceinline__ void amax_merge(float &bv, uint32_t &bi, float v, uint32_t i) {
    if (v > bv || (v == bv && i < bi)) { bv = v; bi = i; }
}

__global__ __launch_bounds__(1024) void k_argmax_part(const float *x, size_t n, size_t per, float *pv, uint32_t *pi) {
    __shared__ float sv[16];
    __shared__ uint32_t si[16];
    float bv = -INFINITY;
    uint32_t bi = 0xFFFFFFFFu;
    size_t s0 = blockIdx.x * per, s1 = s0 + per < n ? s0 + per : n;
    for (size_t i = s0 + threadIdx.x; i < s1; i += blockDim.x) {
        float v = x[i];
        if (v > -INFINITY) amax_merge(bv, bi, v, (uint32_t)i);
    }
    for (int m = 1; m < 64; m <<= 1) {
        float ov = shfl_xor(bv, m);
        uint32_t oi = shfl_xor(bi, m);
        amax_merge(bv, bi, ov, oi);
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0) { sv[wave] = bv; si[wave] = bi; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)(blockDim.x >> 6); w++) amax_merge(bv, bi, sv[w], si[w]);
        pv[blockIdx.x] = bv;
        pi[blockIdx.x] = bi;
    }
}

__global__ void k_argmax_final(const float *pv, const uint32_t *pi, int np, uint32_t *out) {
    float bv = -INFINITY;
    uint32_t bi = 0xFFFFFFFFu;
    for (int i = threadIdx.x; i < np; i += 64) amax_merge(bv, bi, pv[i], pi[i]);
    for (int m = 1; m < 64; m <<= 1) {
        float ov = shfl_xor(bv, m);
        uint32_t oi = shfl_xor(bi, m);
        amax_merge(bv, bi, ov, oi);
    }
    if (threadIdx.x == 0) *out = bi == 0xFFFFFFFFu ? 0u : bi;
}

void launch_argmax(const float *x, size_t n, uint32_t *out_dev, float *scratch, hipStream_t s) {
    const int np = 128;
    size_t per = (n + np - 1) / np;
    float *pv = scratch;
    uint32_t *pi = (uint32_t *)(scratch + np);
    k_argmax_part<<<np, 1024, 0, s>>>(x, n, per, pv, pi);
    k_argmax_final<<<1, 64, 0, s>>>(pv, pi, np, out_dev);
}

// Device-resident greedy loop: next token = argmax, recorded at hist[counter++].
__global__ void k_advance(uint32_t *tok, int *pos, uint32_t *hist, const uint32_t *am) {
    uint32_t t = *am;
    int p = *pos;
    *tok = t;
    if (hist) hist[p] = t;
    *pos = p + 1;
}
void launch_advance(uint32_t *tok_dev, int *counter_dev, uint32_t *hist, const uint32_t *argmax_dev, hipStream_t s) {
    k_advance<<<1, 1, 0, s>>>(tok_dev, counter_dev, hist, argmax_dev);
}

__global__ void k_inc(int *p) { *p = *p + 1; }
void launch_inc(int *p, hipStream_t s) { k_inc<<<1, 1, 0, s>>>(p); }

}  // namespace aotk
