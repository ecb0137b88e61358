// Elementwise, attention, merge and pooling kernels of the encoder pass for
// gfx950, on the ragged packed token layout (request b owns rows
// [start[b], start[b+1]); no padding rows exist).
//
// Semantics follow src/webgpu/ops.ts (cited per kernel). Storage is f16 as in
// the reference's buffers; arithmetic is fp32.
#include <algorithm>

#include "nemo_blocks.h"
#include "nemo_common.h"
#include "nemo_ops.h"
#include "nemo_quant.h"

namespace nemo {

__device__ __forceinline__ float warp_sum(float v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Block-wide sum over blockDim.x (a multiple of 64, at most 1024) threads.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  v = warp_sum(v);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, waves = blockDim.x >> 6;
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float t = lane < waves ? scratch[lane] : 0.f;
  return warp_sum(t);
}

// ---------------------------------------------------------------------------
// Residual add + RMSNorm (src/webgpu/ops.ts:21-56). One workgroup per row,
// 8 values (16 bytes) per thread and pass. The residual delta is either an
// f16 row or the fp32 split-K partial sums of the producing GEMM, summed in
// split order and rounded to f16 (the reference's delta buffer is f16).
// ---------------------------------------------------------------------------

// DELTA = -1: x += f16 delta; S >= 1: x += the sum of S fp32 K-split partials
// (all 2 S loads issued before the first add, added in split order);
// kAnySplits: the same for a run-time count. H16: the partials are f16
// (kEpiPartial16), widened to fp32 before the sum.
constexpr int kAnySplits = 1000;

// Values c .. c + 8 of the row's delta (base = row * hidden).
template <int DELTA, bool H16>
__device__ __forceinline__ void norm_delta8(const void* __restrict__ delta, int splits, size_t base, int c,
                                            size_t slice, float* dv) {
  if constexpr (DELTA > 0 && H16) {
    const uint16_t* p = (const uint16_t*)delta + base + c;
    half8v ph[DELTA];
#pragma unroll
    for (int s = 0; s < DELTA; ++s) ph[s] = *(const half8v*)(p + s * slice);
    float a[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) a[i] = (float)ph[0][i];
#pragma unroll
    for (int s = 1; s < DELTA; ++s)
#pragma unroll
      for (int i = 0; i < 8; ++i) a[i] += (float)ph[s][i];
#pragma unroll
    for (int i = 0; i < 8; ++i) dv[i] = (float)(half_t)a[i];
  } else if constexpr (DELTA > 0) {
    const float* p = (const float*)delta + base + c;
    float4v a, b;
    if constexpr (DELTA == kAnySplits) {
      a = *(const float4v*)p, b = *(const float4v*)(p + 4);
      for (int s = 1; s < splits; ++s) {
        a += *(const float4v*)(p + s * slice);
        b += *(const float4v*)(p + s * slice + 4);
      }
    } else {
      float4v pa[DELTA], pb[DELTA];
#pragma unroll
      for (int s = 0; s < DELTA; ++s) {
        pa[s] = *(const float4v*)(p + s * slice);
        pb[s] = *(const float4v*)(p + s * slice + 4);
      }
      a = pa[0], b = pb[0];
#pragma unroll
      for (int s = 1; s < DELTA; ++s) a += pa[s], b += pb[s];
    }
    const float raw[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int i = 0; i < 8; ++i) dv[i] = (float)(half_t)raw[i];
  } else {
    const half8v d16 = *(const half8v*)((const uint16_t*)delta + base + c);
#pragma unroll
    for (int i = 0; i < 8; ++i) dv[i] = (float)d16[i];
  }
}

// f16(x * inv * w) of 8 values.
__device__ __forceinline__ half8v norm_scale8(half8v xv, float inv, const float4v& w0, const float4v& w1) {
  const float wv[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
  half8v o;
#pragma unroll
  for (int i = 0; i < 8; ++i) o[i] = (half_t)(((float)xv[i] * inv) * wv[i]);
  return o;
}

// One row: fetch(c, sum) returns the row's stored values c .. c + 8 and adds
// the squares of their unrounded forms to `sum`, in order and each with one
// fmaf: left to contraction, s + v * v may round either product of the first
// two values, and every later layer of a pass differs with the choice. A row
// of up to 8 values per thread (hidden 2048 and below) stays in registers
// between the two passes, its weights loaded beside it; a longer one is read
// back from xrow, which fetch writes (so xrow is not __restrict__).
template <typename Fetch>
__device__ __forceinline__ void norm_row(Fetch&& fetch, const uint16_t* xrow, const float* __restrict__ w,
                                         uint16_t* __restrict__ orow, int hidden, float eps, float* scratch) {
  const int c0 = threadIdx.x * 8, step = blockDim.x * 8;
  float sum = 0.f;
  if (hidden <= step) {
    half8v xv = {};
    float4v w0 = {}, w1 = {};
    if (c0 < hidden) {
      w0 = *(const float4v*)(w + c0), w1 = *(const float4v*)(w + c0 + 4);
      xv = fetch(c0, sum);
    }
    const float total = block_sum(sum, scratch);
    const float inv = 1.0f / sqrtf(total / (float)hidden + eps);
    if (c0 < hidden) *(half8v*)(orow + c0) = norm_scale8(xv, inv, w0, w1);
    return;
  }
  for (int c = c0; c < hidden; c += step) (void)fetch(c, sum);
  const float total = block_sum(sum, scratch);
  const float inv = 1.0f / sqrtf(total / (float)hidden + eps);
  for (int c = c0; c < hidden; c += step)
    *(half8v*)(orow + c) = norm_scale8(*(const half8v*)(xrow + c), inv, *(const float4v*)(w + c), *(const float4v*)(w + c + 4));
}

template <int DELTA, bool H16 = false>
__global__ __launch_bounds__(256) void rmsnorm_kernel(uint16_t* x, const void* __restrict__ delta, int splits,
                                                      int rows, const float* __restrict__ w,
                                                      uint16_t* __restrict__ out, int hidden, float eps) {
  __shared__ float scratch[16];
  const size_t base = (size_t)blockIdx.x * hidden, slice = (size_t)rows * hidden;
  auto fetch = [&](int c, float& sum) {
    const half8v xv = *(const half8v*)(x + base + c);
    float dv[8];
    norm_delta8<DELTA, H16>(delta, splits, base, c, slice, dv);
    half8v stored;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float v = (float)xv[i] + dv[i];
      sum = fmaf(v, v, sum);  // the unrounded sum, as ops.ts:39-40
      stored[i] = (half_t)v;
    }
    *(half8v*)(x + base + c) = stored;
    return stored;
  };
  norm_row(fetch, x + base, w, out + base, hidden, eps, scratch);
}

// Embedding lookup (src/webgpu/ops.ts:680-710) and the first layer's RMSNorm
// of the same row in one launch (two launches took 6.1 us for one 15-token
// request and 36 us for 12,000 tokens, one takes 3.8 and 28: the row is not
// read back).
template <int TABLE>
__global__ __launch_bounds__(256) void embed_norm_kernel(const uint32_t* __restrict__ ids, int padded_seq, Ragged rows,
                                                         const void* __restrict__ table, int vocab, uint16_t* x,
                                                         const float* __restrict__ w, uint16_t* __restrict__ out,
                                                         int hidden, float eps) {
  __shared__ float scratch[16];
  const int t = blockIdx.x;
  const int b = ragged_find(rows, t);
  uint32_t id = ids[(size_t)b * padded_seq + (t - rows.start[b])];
  if (id >= (uint32_t)vocab) id = 0;  // out-of-range ids are rejected on the host; never read past the table
  uint16_t* xrow = x + (size_t)t * hidden;
  auto fetch = [&](int c, float& sum) {
    half8v v;
    if constexpr (TABLE == kF16) {
      v = *(const half8v*)((const uint16_t*)table + (size_t)id * hidden + c);
    } else {
      // Q6_K row, f16(d * scale * (q - 32)) (ops.ts:689-703): 8 values of one
      // quadrant Q of half h of a 256-value block, from lane l on.
      const uint8_t* p = (const uint8_t*)table + ((size_t)id * (hidden / 256) + (c >> 8)) * 210;
      const int h = (c >> 7) & 1, Q = (c >> 5) & 3, l = c & 31;
      const uint16_t* ql = (const uint16_t*)(p + 64 * h + 32 * (Q & 1) + l);
      const uint16_t* qh = (const uint16_t*)(p + 128 + 32 * h + l);
      const float dsc = h2f(*(const uint16_t*)(p + 208)) * (float)(int8_t)p[192 + 8 * h + 2 * Q + (l >> 4)];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const uint32_t low = ((uint32_t)ql[e >> 1] >> (8 * (e & 1) + (Q >= 2 ? 4 : 0))) & 15u;
        const uint32_t high = ((uint32_t)qh[e >> 1] >> (8 * (e & 1) + 2 * Q)) & 3u;
        v[e] = (half_t)(dsc * (float)((int)(low | (high << 4)) - 32));
      }
    }
    *(half8v*)(xrow + c) = v;
#pragma unroll
    for (int i = 0; i < 8; ++i) sum = fmaf((float)v[i], (float)v[i], sum);
    return v;
  };
  norm_row(fetch, xrow, w, out + (size_t)t * hidden, hidden, eps, scratch);
}

hipError_t launch_embed_norm(const uint32_t* ids, int padded_seq, const Ragged& rows, int table_type,
                             const void* table, int hidden, int vocab, uint16_t* x, const float* w,
                             uint16_t* normalized, float eps, hipStream_t stream) {
  const int total = rows.start[rows.count];
  if (total <= 0) return hipSuccess;
  if (table_type == kF16)
    embed_norm_kernel<kF16><<<total, 256, 0, stream>>>(ids, padded_seq, rows, table, vocab, x, w, normalized, hidden,
                                                       eps);
  else if (table_type == kQ6_K)
    embed_norm_kernel<kQ6_K><<<total, 256, 0, stream>>>(ids, padded_seq, rows, table, vocab, x, w, normalized, hidden,
                                                        eps);
  else
    return hipErrorInvalidValue;
  return hipGetLastError();
}

hipError_t launch_rmsnorm(uint16_t* x, const uint16_t* delta, const float* w, uint16_t* normalized, int rows,
                          int hidden, float eps, hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  rmsnorm_kernel<-1><<<rows, 256, 0, stream>>>(x, delta, 1, rows, w, normalized, hidden, eps);
  return hipGetLastError();
}

hipError_t launch_rmsnorm_partials(uint16_t* x, const float* partials, int splits, const float* w,
                                   uint16_t* normalized, int rows, int hidden, float eps, hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
  if (splits < 1) return hipErrorInvalidValue;
#define NEMO_NORM(S) rmsnorm_kernel<S><<<rows, 256, 0, stream>>>(x, partials, splits, rows, w, normalized, hidden, eps)
  switch (splits) {
    case 1: NEMO_NORM(1); break;
    case 2: NEMO_NORM(2); break;
    case 3: NEMO_NORM(3); break;
    case 4: NEMO_NORM(4); break;
    case 6: NEMO_NORM(6); break;
    case 8: NEMO_NORM(8); break;
    case 12: NEMO_NORM(12); break;
    case 16: NEMO_NORM(16); break;
    default: NEMO_NORM(kAnySplits); break;
  }
#undef NEMO_NORM
  return hipGetLastError();
}

hipError_t launch_rmsnorm_partials16(uint16_t* x, const uint16_t* partials, int splits, const float* w,
                                     uint16_t* normalized, int rows, int hidden, float eps, hipStream_t stream) {
  if (rows <= 0) return hipSuccess;
#define NEMO_NORM16(S) \
  rmsnorm_kernel<S, true><<<rows, 256, 0, stream>>>(x, partials, splits, rows, w, normalized, hidden, eps)
  switch (splits) {
    case 2: NEMO_NORM16(2); break;
    case 3: NEMO_NORM16(3); break;
    case 4: NEMO_NORM16(4); break;
    default: return hipErrorInvalidValue;
  }
#undef NEMO_NORM16
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Pairwise RoPE (src/webgpu/ops.ts:168-193): (e, o) -> (e c - o s, e s + o c)
// with (c, s) = table[position][pair], on 8 consecutive values of a head (4
// pairs) at a time. The attention kernel applies it as it loads queries and
// keys from the QKV projection; rope_kernel writes the rotated heads out
// (one workgroup per token) for inspection of the stage.
// ---------------------------------------------------------------------------

// v = values 2p0 .. 2p0 + 7 of a head; (a, b) = the table's (c, s) of its 4
// pairs (table row + 2 p0, 8 floats).
__device__ __forceinline__ half8v rope8(half8v v, float4v a, float4v b) {
  const float c[4] = {a[0], a[2], b[0], b[2]}, sn[4] = {a[1], a[3], b[1], b[3]};
  half8v r;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const float e = (float)v[2 * j], o = (float)v[2 * j + 1];
    r[2 * j] = (half_t)(e * c[j] - o * sn[j]);
    r[2 * j + 1] = (half_t)(e * sn[j] + o * c[j]);
  }
  return r;
}
__device__ __forceinline__ half8v rope8(half8v v, const float* __restrict__ cs) {
  return rope8(v, *(const float4v*)cs, *(const float4v*)(cs + 4));
}

__global__ __launch_bounds__(256) void rope_kernel(const uint16_t* __restrict__ qkv, int qkv_stride, Ragged rows,
                                                   const float* __restrict__ table, int q_heads, int kv_heads,
                                                   int head_dim, uint16_t* __restrict__ q, uint16_t* __restrict__ k) {
  const int t = blockIdx.x;
  const int b = ragged_find(rows, t);
  const int pos = t - rows.start[b];
  const int chunks = head_dim / 8, total = (q_heads + kv_heads) * chunks;
  const float* trow = table + (size_t)pos * head_dim;
  for (int i = threadIdx.x; i < total; i += blockDim.x) {
    const int head = i / chunks, d = 8 * (i - head * chunks);
    const half8v r = rope8(*(const half8v*)(qkv + (size_t)t * qkv_stride + head * head_dim + d), trow + d);
    if (head < q_heads)
      *(half8v*)(q + ((size_t)t * q_heads + head) * head_dim + d) = r;
    else
      *(half8v*)(k + ((size_t)t * kv_heads + (head - q_heads)) * head_dim + d) = r;
  }
}

hipError_t launch_rope(const uint16_t* qkv, int qkv_stride, const Ragged& rows, const float* table, int q_heads,
                       int kv_heads, int head_dim, uint16_t* q, uint16_t* k, hipStream_t stream) {
  const int total = rows.start[rows.count];
  if (total <= 0) return hipSuccess;
  if (head_dim % 8) return hipErrorInvalidValue;
  rope_kernel<<<total, 256, 0, stream>>>(qkv, qkv_stride, rows, table, q_heads, kv_heads, head_dim, q, k);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Bidirectional GQA flash attention on MFMA (src/webgpu/ops.ts:213-293,
// 295-362), reading queries, keys and values from the QKV projection [t,
// (Hq + 2 Hkv) hd] and rotating queries and keys (RoPE, position = row
// within the request) as it loads them. For request b with n valid rows,
// query i attends keys
// 0, s, 2s, ... < n (s = key_stride if n > stride_threshold, else 1) with
// scores q.k * head_dim^-1/2 * temperature(i), temperature = 1 + 0.1
// ln(floor(i / 16384) + 1) for i >= 16384 (ops.ts:241); online softmax in
// fp32, output f16.
//
// Workgroup = one request, one KV head, 32 queries; wave w handles query
// head kv_head * group + w, so the staged K/V tiles serve the whole GQA
// group. Scores are computed transposed, S^T = K Q^T (32 keys x 32 queries
// per v_mfma_f32_32x32x16_f16), so lane l always holds query l%32: the
// softmax max/sum are per-lane scalars (one cross-half exchange), and the
// rescale of the output accumulators is a per-lane multiply. The output is
// accumulated transposed too, O^T = V^T P^T, with V staged transposed in LDS
// and P fed from the score registers: the MFMA's k index is mapped to the
// keys a lane holds (the key order of a sum is free; A and B agree on it).
// ---------------------------------------------------------------------------

constexpr int kAttnQ = 32, kAttnKeys = 32;

__device__ __forceinline__ int attn_keys(int n, int stride_threshold, int key_stride_long) {
  const int s = n > stride_threshold ? key_stride_long : 1;
  return (n + s - 1) / s;
}

constexpr int kAttnLongWaves = 4;
// Workgroups of a request and KV head: 4 (32-query tile, head) pairs each.
__host__ __device__ inline int attn_long_workgroups(int n, int group) {
  return (group * ((n + kAttnQ - 1) / kAttnQ) + kAttnLongWaves - 1) / kAttnLongWaves;
}
typedef __attribute__((address_space(3))) void attn_lds_void;

// Long requests: one pass per layer writes each request's attended keys,
// rotated, and its values transposed, in blocks of 32 keys (request b's from
// block sum over earlier requests of ceil(keys / 32), zero past its last key),
// each the LDS image that attention_long_kernel copies as it is:
//   K_s  [kv head][block][key][16-byte chunk c at c ^ attn_kswz(key)]
//   V^T_s [kv head][block][d][4 chunks of 8 keys, chunk q at q ^ attn_vswz(d)],
// chunk q = 2 c2 + hl holding the keys 16 c2 + 8 (e / 4) + 4 hl + e % 4, e =
// 0..7, that lane half hl's score registers 8 c2 + e hold. The swizzles spread
// the rows that one fragment read touches over distinct banks. Workgroup = 32
// keys of one kv head.
template <int HD>
__device__ __forceinline__ int attn_kswz(int key) {
  return HD == 128 ? key & 15 : (key & 7) ^ ((key >> 3) & 1);
}
__device__ __forceinline__ int attn_vswz(int d) { return (((d >> 1) ^ (d >> 3)) & 1) | (((d >> 2) & 1) << 1); }

template <int HD>
__global__ __launch_bounds__(256) void attention_prep_kernel(const uint16_t* __restrict__ qkv, int qkv_stride,
                                                             const float* __restrict__ table, Ragged rows,
                                                             int q_heads, int kv_heads, int stride_threshold,
                                                             int key_stride_long, int keys_cap,
                                                             uint16_t* __restrict__ ks, uint16_t* __restrict__ vts) {
  __shared__ __attribute__((aligned(16))) half_t sv[kAttnKeys * (HD + 8)];
  const int kvh = blockIdx.x % kv_heads, block = blockIdx.x / kv_heads;
  int b = 0, blk = block;
  for (; b < rows.count; ++b) {
    const int blocks = (attn_keys(rows.start[b + 1] - rows.start[b], stride_threshold, key_stride_long) + 31) / 32;
    if (blk < blocks) break;
    blk -= blocks;
  }
  if (b >= rows.count) return;
  const int row0 = rows.start[b], n = rows.start[b + 1] - row0;
  const int key_stride = n > stride_threshold ? key_stride_long : 1;
  const int n_keys = (n + key_stride - 1) / key_stride;
  const size_t image = ((size_t)kvh * keys_cap + kAttnKeys * block) * HD;  // this block in either buffer
  const uint16_t* kbase = qkv + (q_heads + kvh) * HD;
  const uint16_t* vbase = qkv + (q_heads + kv_heads + kvh) * HD;
  for (int i = threadIdx.x; i < kAttnKeys * HD / 8; i += blockDim.x) {
    const int j = i / (HD / 8), c = (i % (HD / 8)) * 8, key = kAttnKeys * blk + j;
    half8v kv = {}, vv = {};
    if (key < n_keys) {
      const int kpos = key * key_stride;
      const size_t trow = (size_t)(row0 + kpos) * qkv_stride;
      kv = rope8(*(const half8v*)(kbase + trow + c), table + (size_t)kpos * HD + c);
      vv = *(const half8v*)(vbase + trow + c);
    }
    *(half8v*)(ks + image + j * HD + 8 * ((c >> 3) ^ attn_kswz<HD>(j))) = kv;
    *(half8v*)&sv[j * (HD + 8) + c] = vv;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < HD * kAttnKeys / 8; i += blockDim.x) {
    const int d = i / (kAttnKeys / 8), q = i % (kAttnKeys / 8);
    half8v col;
#pragma unroll
    for (int e = 0; e < 8; ++e) col[e] = sv[(16 * (q >> 1) + 8 * (e >> 2) + 4 * (q & 1) + (e & 3)) * (HD + 8) + d];
    *(half8v*)(vts + image + d * kAttnKeys + 8 * (q ^ attn_vswz(d))) = col;
  }
}

// A wave's 32 queries of one head: query l%32 in lane l, whose half hl = l/32
// holds d 32db + 8j + 4hl + 0..3 in registers 4j.. of o[db], and the sum of its
// own keys' probabilities. m: the query's reference maximum (log2 units,
// scaled).
template <int HD>
struct AttnRows {
  static constexpr int DB = HD / 32;  // 32-wide d blocks of the output
  float16v o[DB];
  float m = -INFINITY, lsum = 0.f;

  __device__ __forceinline__ AttnRows() {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[db][r] = 0.f;
  }

  // The probabilities of one block of 32 keys, as the B operands of its two
  // 16-key chunks: s register r is the score of key 8(r/4) + 4hl + r%4, of
  // which the first `valid` exist.
  //
  // Probabilities are taken against a reference maximum m that is raised
  // only when a query's block maximum exceeds it by more than 2^8 (a wave
  // vote): p = 2^(s - m) <= 256 then, exact enough in f16 and far from
  // overflow in the fp32 sums, and the common block needs no cross-lane
  // exchange, no rescale of the accumulators and no 2^(m - m') of its own.
  // The result is the softmax all the same: numerator and denominator share
  // the reference.
  __device__ __forceinline__ void probabilities(float16v s, float scale2, int valid, int hl, half8v (&pb)[2]) {
    if (valid < kAttnKeys) {  // the request's last keys: mask past its end
      asm volatile("");       // keeps this rare path a branch (not computed and selected every block)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        if (8 * (r >> 2) + 4 * hl + (r & 3) >= valid) s[r] = -INFINITY;
    }
    float bm = s[0];
#pragma unroll
    for (int r = 1; r < 16; ++r) bm = fmaxf(bm, s[r]);
    bm *= scale2;  // scale2 > 0: the maximum of the scaled scores
    if (__builtin_amdgcn_ballot_w64(bm > m + 8.0f)) {
      asm volatile("");
      const float mn = fmaxf(m, fmaxf(bm, __shfl_xor(bm, 32, 64)));
      const float alpha = __builtin_amdgcn_exp2f(m - mn);
      lsum *= alpha;
#pragma unroll
      for (int db = 0; db < DB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
      m = mn;
    }
    float p[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      // v_exp_f32 itself: results below 2^-126 (flushed) add nothing to the sums
      p[r] = __builtin_amdgcn_exp2f(fmaf(s[r], scale2, -m));
      lsum += p[r];
    }
    pb[0] = to_half8(p);
    pb[1] = to_half8(p + 8);
  }

  __device__ __forceinline__ void store(uint16_t* __restrict__ op, int hl) {
    const float inv = 1.0f / lsum;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const half4v hv = {(half_t)(o[db][4 * j] * inv), (half_t)(o[db][4 * j + 1] * inv),
                           (half_t)(o[db][4 * j + 2] * inv), (half_t)(o[db][4 * j + 3] * inv)};
        *(half4v*)(op + 32 * db + 8 * j + 4 * hl) = hv;
      }
  }
};

// Query fragments of one head (16-wide d chunks), rotated; and the scores'
// factor in log2 units.
template <int HD>
__device__ __forceinline__ void attn_queries(const uint16_t* __restrict__ qkv, int qkv_stride,
                                             const float* __restrict__ table, int row0, int qpos, int h, int hl,
                                             half8v (&qf)[HD / 16]) {
  const uint16_t* qp = qkv + (size_t)(row0 + qpos) * qkv_stride + h * HD + 8 * hl;
  const float* cs = table + (size_t)qpos * HD + 8 * hl;
#pragma unroll
  for (int c = 0; c < HD / 16; ++c) qf[c] = rope8(*(const half8v*)(qp + 16 * c), cs + 16 * c);
}
template <int HD>
__device__ __forceinline__ float attn_scale2(int qi) {
  const float temperature = qi >= 16384 ? logf(floorf((float)qi / 16384.0f) + 1.0f) * 0.1f + 1.0f : 1.0f;
  return (1.0f / sqrtf((float)HD)) * temperature * 1.4426950408889634f;
}

// Requests of at most one staging round of keys (and any when the key images
// are not there): keys and values staged from the QKV projection.
template <int HD>
__global__ __launch_bounds__(512) void attention_kernel(const uint16_t* __restrict__ qkv, int qkv_stride,
                                                        const float* __restrict__ table, Ragged rows, int q_heads,
                                                        int kv_heads, int stride_threshold, int key_stride_long,
                                                        int sb_keys, uint16_t* __restrict__ out) {
  constexpr int KP = HD + 8;  // padded K row (halves)
  constexpr int DC = HD / 16; // 16-wide d chunks of the score MFMAs
  constexpr int DB = HD / 32; // 32-wide d blocks of the output
  // sb_keys (a multiple of 32) keys are staged per round: sK [sb_keys][KP],
  // sVt [HD][VP].
  extern __shared__ __attribute__((aligned(16))) uint8_t attn_lds[];
  const int VP = sb_keys + 8;
  half_t* sK = (half_t*)attn_lds;
  half_t* sVt = sK + sb_keys * KP;
  const int kvh = blockIdx.x % kv_heads;  // fastest: a KV head's workgroups share an XCD's L2
  int b = 0, tile = blockIdx.x / kv_heads;
  for (; b < rows.count; ++b) {
    const int tiles = (rows.start[b + 1] - rows.start[b] + kAttnQ - 1) / kAttnQ;
    if (tile < tiles) break;
    tile -= tiles;
  }
  if (b >= rows.count) return;
  const int row0 = rows.start[b];
  const int n = rows.start[b + 1] - row0;
  const int group = q_heads / kv_heads;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, hl = lane >> 5;
  const int h = kvh * group + wave;
  const int qi = tile * kAttnQ + (lane & 31);
  const int key_stride = n > stride_threshold ? key_stride_long : 1;
  const int n_keys = (n + key_stride - 1) / key_stride;
  const float scale2 = attn_scale2<HD>(qi);
  half8v qf[DC];
  attn_queries<HD>(qkv, qkv_stride, table, row0, min(qi, n - 1), h, hl, qf);
  const uint16_t* kbase = qkv + (q_heads + kvh) * HD;
  const uint16_t* vbase = qkv + (q_heads + kv_heads + kvh) * HD;
  AttnRows<HD> acc;

  // The block of staged keys from kb; keys at or past `staged` are masked.
  auto block = [&](int kb, int staged) {
    float16v s = {};
#pragma unroll
    for (int c = 0; c < DC; ++c) {
      const half8v a = *(const half8v*)&sK[(kb + (lane & 31)) * KP + 16 * c + 8 * hl];
      s = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qf[c], s, 0, 0, 0);
    }
    half8v pb[2];
    acc.probabilities(s, scale2, staged - kb, hl, pb);
    // O^T += V^T P^T over two 16-key chunks: MFMA k slot 8hl + e of chunk c2
    // is key 16c2 + 8(e/4) + 4hl + e%4 = score register 8c2 + e.
#pragma unroll
    for (int c2 = 0; c2 < 2; ++c2)
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const half_t* vr = &sVt[(32 * db + (lane & 31)) * VP + kb + 16 * c2 + 4 * hl];
        const half4v v0 = *(const half4v*)vr;
        const half4v v1 = *(const half4v*)(vr + 8);
        const half8v a = {v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
        acc.o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, pb[c2], acc.o[db], 0, 0, 0);
      }
  };
  for (int sb = 0; sb < n_keys; sb += sb_keys) {
    const int staged = min(sb_keys, n_keys - sb);
    __syncthreads();
    // 16-byte chunks of the staged keys (rows past `staged` up to the
    // next multiple of 32 are zero), in batches of 4 per thread with every
    // load of a batch issued before the first is used.
    const int chunks = (staged + 31) / 32 * 32 * HD / 8;
    for (int i0 = threadIdx.x; i0 < chunks; i0 += 4 * blockDim.x) {
      half8v kr[4], vr[4];
      float4v ca[4], cb[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = i0 + u * blockDim.x, j = i / (HD / 8), c = (i % (HD / 8)) * 8;
        kr[u] = half8v{};
        vr[u] = half8v{};
        ca[u] = cb[u] = float4v{0.f, 0.f, 0.f, 0.f};
        if (i < chunks && j < staged) {
          const int kpos = (sb + j) * key_stride;
          const size_t trow = (size_t)(row0 + kpos) * qkv_stride;
          kr[u] = *(const half8v*)(kbase + trow + c);
          vr[u] = *(const half8v*)(vbase + trow + c);
          const float* cs = table + (size_t)kpos * HD + c;
          ca[u] = *(const float4v*)cs;
          cb[u] = *(const float4v*)(cs + 4);
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int i = i0 + u * blockDim.x, j = i / (HD / 8), c = (i % (HD / 8)) * 8;
        if (i < chunks) {
          *(half8v*)&sK[j * KP + c] = rope8(kr[u], ca[u], cb[u]);
#pragma unroll
          for (int e = 0; e < 8; ++e) sVt[(c + e) * VP + j] = vr[u][e];
        }
      }
    }
    __syncthreads();
    for (int kb = 0; kb < staged; kb += kAttnKeys) block(kb, staged);
  }
  acc.lsum += __shfl_xor(acc.lsum, 32, 64);  // the two halves' keys (same references)
  if (qi < n) acc.store(out + ((size_t)(row0 + qi) * q_heads + h) * HD, hl);
}

// Longer requests, on the key images of attention_prep_kernel. Workgroup = 4
// waves = 4 consecutive (32-query tile, head of the group) pairs of one
// request and KV head; 64 keys per round (two images of 32), copied global ->
// LDS in two stages, one barrier per round, the copies of round r + 1 in
// flight under round r. The two blocks' score chains are independent, and one
// block's exponentials run under the other's MFMAs.
//
// Bound by the vector ALU (exponentials, maxima and conversions; active 62 % of
// the cycles at 5000 tokens and 32 heads of 64) and the MFMAs (31 %), which
// take turns on a SIMD of few waves; the LDS is active 16 %, without
// conflicts. What it replaced staged 32 keys per barrier through registers for
// one workgroup of `group` waves (3 at 24 heads of 128: 6 waves on a CU, on 2
// of its SIMDs 2): 8 x 1500 tokens, 24 heads of 128, 458 -> 277 us a layer; 5000
// tokens, 32 heads of 64, every third key, 109 -> 101, 3200 64 -> 53 (same
// bits). The KV head runs fastest in the grid, so with 8 of them each XCD's L2
// holds the images of one.
template <int HD>
__global__ __launch_bounds__(256, HD == 128 ? 2 : 4)
void attention_long_kernel(const uint16_t* __restrict__ qkv, int qkv_stride, const float* __restrict__ table,
                           Ragged rows, int q_heads, int kv_heads, int stride_threshold, int key_stride_long,
                           const uint16_t* __restrict__ ks, const uint16_t* __restrict__ vts, int keys_cap,
                           uint16_t* __restrict__ out) {
  constexpr int DC = HD / 16, DB = HD / 32;
  constexpr int IMG = 2 * kAttnKeys * HD;  // bytes of an image of 32 keys
  __shared__ __attribute__((aligned(16))) uint8_t lds[2][2][2 * IMG];  // [stage][block]: K, then V^T
  const int group = q_heads / kv_heads;
  const int kvh = blockIdx.x % kv_heads;
  int b = 0, wg = blockIdx.x / kv_heads, koff = 0;  // koff: the request's first key in the images
  for (; b < rows.count; ++b) {
    const int n = rows.start[b + 1] - rows.start[b];
    const int wgs = attn_long_workgroups(n, group);
    if (wg < wgs) break;
    wg -= wgs;
    koff += kAttnKeys * ((attn_keys(n, stride_threshold, key_stride_long) + kAttnKeys - 1) / kAttnKeys);
  }
  if (b >= rows.count) return;
  const int row0 = rows.start[b];
  const int n = rows.start[b + 1] - row0;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), hl = lane >> 5;
  const int item = kAttnLongWaves * wg + wave;
  const bool active = item < group * ((n + kAttnQ - 1) / kAttnQ);  // uniform in the wave
  const int tile = active ? item / group : 0;
  const int h = kvh * group + item % group;
  const int qi = tile * kAttnQ + (lane & 31);
  const int n_keys = attn_keys(n, stride_threshold, key_stride_long);
  const int blocks = (n_keys + kAttnKeys - 1) / kAttnKeys, rounds = (blocks + 1) >> 1;

  const size_t first = ((size_t)kvh * keys_cap + koff) * HD;
  auto stage = [&](int r) {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      if (2 * r + u >= blocks) break;
      const size_t image = first + (size_t)(2 * r + u) * kAttnKeys * HD;
      uint8_t* dst = lds[r & 1][u];
#pragma unroll
      for (int i = 0; i < HD / 64; ++i) {  // 1 KB per instruction
        const int at = 1024 * (HD / 64 * wave + i);
        __builtin_amdgcn_global_load_lds((const void*)(ks + image + at / 2 + 8 * lane), (attn_lds_void*)(dst + at), 16, 0, 0);
        __builtin_amdgcn_global_load_lds((const void*)(vts + image + at / 2 + 8 * lane),
                                         (attn_lds_void*)(dst + IMG + at), 16, 0, 0);
      }
    }
  };
  stage(0);
  const float scale2 = attn_scale2<HD>(qi);
  half8v qf[DC];
  attn_queries<HD>(qkv, qkv_stride, table, row0, min(qi, n - 1), h, hl, qf);
  AttnRows<HD> acc;
  const int krow = (lane & 31) * HD * 2, ksw = attn_kswz<HD>(lane & 31);
  const int vrow = IMG + (lane & 31) * kAttnKeys * 2, vsw = attn_vswz(lane & 31);  // rows 32 apart share the swizzle
  auto score = [&](const uint8_t* img, int c, float16v& s) {
    const half8v a = *(const half8v*)(img + krow + 16 * ((2 * c + hl) ^ ksw));
    s = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, qf[c], s, 0, 0, 0);
  };
  auto values = [&](const uint8_t* img, const half8v (&pb)[2]) {
#pragma unroll
    for (int c2 = 0; c2 < 2; ++c2)
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        const half8v a = *(const half8v*)(img + vrow + db * 32 * kAttnKeys * 2 + 16 * ((2 * c2 + hl) ^ vsw));
        acc.o[db] = __builtin_amdgcn_mfma_f32_32x32x16_f16(a, pb[c2], acc.o[db], 0, 0, 0);
      }
  };
  for (int r = 0; r < rounds; ++r) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();  // round r has landed, and every wave has left the other stage
    if (r + 1 < rounds) stage(r + 1);
    if (!active) continue;
    const uint8_t* i0 = lds[r & 1][0];
    const uint8_t* i1 = lds[r & 1][1];
    const int valid = n_keys - 2 * kAttnKeys * r;
    half8v pb[2];
    float16v s0 = {}, s1 = {};
    if (valid > kAttnKeys) {
#pragma unroll
      for (int c = 0; c < DC; ++c) {
        score(i0, c, s0);
        score(i1, c, s1);
      }
      acc.probabilities(s0, scale2, kAttnKeys, hl, pb);
      values(i0, pb);
      acc.probabilities(s1, scale2, valid - kAttnKeys, hl, pb);
      values(i1, pb);
    } else {
#pragma unroll
      for (int c = 0; c < DC; ++c) score(i0, c, s0);
      acc.probabilities(s0, scale2, valid, hl, pb);
      values(i0, pb);
    }
  }
  acc.lsum += __shfl_xor(acc.lsum, 32, 64);  // the two halves' keys (same references)
  if (active && qi < n) acc.store(out + ((size_t)(row0 + qi) * q_heads + h) * HD, hl);
}

int attention_prep_keys(const Ragged& rows, int stride_threshold, int key_stride) {
  int keys = 0;
  for (int b = 0; b < rows.count; ++b) {
    const int n = rows.start[b + 1] - rows.start[b];
    const int s = n > stride_threshold ? key_stride : 1;
    keys += kAttnKeys * (((n + s - 1) / s + kAttnKeys - 1) / kAttnKeys);
  }
  return keys;
}

hipError_t launch_attention(const uint16_t* qkv, int qkv_stride, const float* rope_table, const Ragged& rows,
                            int q_heads, int kv_heads, int head_dim, int stride_threshold, int key_stride, uint16_t* out,
                            hipStream_t stream, uint16_t* ks, uint16_t* vts, int keys_cap) {
  int tiles = 0, wgs = 0, longest_keys = 0;
  const int group = kv_heads > 0 ? q_heads / kv_heads : 0;
  if (group < 1 || group > 8 || q_heads % kv_heads) return hipErrorInvalidValue;
  if (head_dim != 64 && head_dim != 128) return hipErrorInvalidValue;
  for (int b = 0; b < rows.count; ++b) {
    const int n = rows.start[b + 1] - rows.start[b];
    tiles += (n + kAttnQ - 1) / kAttnQ;
    wgs += attn_long_workgroups(n, group);
    const int s = n > stride_threshold ? key_stride : 1;
    longest_keys = std::max(longest_keys, (n + s - 1) / s);
  }
  if (tiles == 0) return hipSuccess;
  if (ks != nullptr) {
    const int keys = attention_prep_keys(rows, stride_threshold, key_stride);
    if (!vts || keys > keys_cap || keys_cap % kAttnKeys) return hipErrorInvalidValue;
    const unsigned pgrid = (unsigned)kv_heads * (keys / kAttnKeys), grid = (unsigned)kv_heads * wgs;
    auto launch = [&](auto prep, auto attend) {
      prep<<<pgrid, 256, 0, stream>>>(qkv, qkv_stride, rope_table, rows, q_heads, kv_heads, stride_threshold,
                                      key_stride, keys_cap, ks, vts);
      attend<<<grid, 64 * kAttnLongWaves, 0, stream>>>(qkv, qkv_stride, rope_table, rows, q_heads, kv_heads,
                                                       stride_threshold, key_stride, ks, vts, keys_cap, out);
    };
    if (head_dim == 64) launch(attention_prep_kernel<64>, attention_long_kernel<64>);
    else launch(attention_prep_kernel<128>, attention_long_kernel<128>);
    return hipGetLastError();
  }
  const unsigned grid = (unsigned)kv_heads * tiles;
  // Keys staged per round: every key of the pass's longest request when
  // they fit in ~72 KB of LDS (one round of loads and barriers instead of one
  // per 32 keys).
  const int cap = attn_round_keys(head_dim);
  const int sb = std::min(cap, (longest_keys + kAttnKeys - 1) / kAttnKeys * kAttnKeys);
  const int lds = 2 * (sb * (head_dim + 8) + head_dim * (sb + 8));
  auto launch = [&](auto hd) {
    constexpr auto kernel = attention_kernel<decltype(hd)::value>;
    allow_lds<kernel>(2 * (cap * (head_dim + 8) + head_dim * (cap + 8)));
    kernel<<<grid, 64 * group, lds, stream>>>(qkv, qkv_stride, rope_table, rows, q_heads, kv_heads, stride_threshold,
                                              key_stride, sb, out);
  };
  if (head_dim == 64) launch(std::integral_constant<int, 64>{});
  else launch(std::integral_constant<int, 128>{});
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Adjacent-state token merge (src/webgpu/ops.ts:629-660): output position 0
// is source row 0 (BOS); position p > 0 averages source rows [start, end) with
// start = 1 + (p-1)(S-1)/(T-1), end = max(1 + p(S-1)/(T-1), start+1) min S.
// One workgroup per output row and stream: the normalized stream and, with
// blockIdx.y = 1, the residual stream in the same launch (10 rows: two
// launches 5.5 us, one 3.3).
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(256) void merge_kernel(const uint16_t* __restrict__ in0, const uint16_t* __restrict__ in1,
                                                    Ragged src, Ragged dst, int hidden, uint16_t* __restrict__ out0,
                                                    uint16_t* __restrict__ out1) {
  const uint16_t* in = blockIdx.y ? in1 : in0;
  uint16_t* out = blockIdx.y ? out1 : out0;
  const int t = blockIdx.x;
  const int b = ragged_find(dst, t);
  const int p = t - dst.start[b];
  const int S = src.start[b + 1] - src.start[b];
  const int T = dst.start[b + 1] - dst.start[b];
  int start = 0, end = 1;
  if (p > 0 && T > 1) {
    const int st = S - 1, tt = T - 1;
    start = 1 + (int)(((int64_t)(p - 1) * st) / tt);
    end = 1 + (int)(((int64_t)p * st) / tt);
    end = max(end, start + 1);
    end = min(end, S);
  }
  const float inv = 1.0f / (float)(end - start);
  for (int c = threadIdx.x * 8; c < hidden; c += blockDim.x * 8) {
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    for (int r = start; r < end; ++r) {
      const half8v v = *(const half8v*)(in + (size_t)(src.start[b] + r) * hidden + c);
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[e] += (float)v[e];
    }
    half8v o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = (half_t)(acc[e] * inv);
    *(half8v*)(out + (size_t)t * hidden + c) = o;
  }
}

hipError_t launch_merge(const uint16_t* norm, const uint16_t* x, const Ragged& src, const Ragged& dst, int hidden,
                        uint16_t* norm_out, uint16_t* x_out, hipStream_t stream) {
  const int total = dst.start[dst.count];
  if (total <= 0) return hipSuccess;
  merge_kernel<<<dim3(total, x ? 2 : 1), 256, 0, stream>>>(norm, x, src, dst, hidden, norm_out, x_out);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// Mean pool + L2 normalise (src/webgpu/ops.ts:596-615), in two kernels so a
// request is read by many CUs:
//  * pool_mean_kernel, grid (hidden / 32, batch): a workgroup owns 32 columns
//    of one request; thread (g, p) sums 8 columns (16-byte loads) of rows p,
//    p + 32, ... in order, and the 32 row phases are added in phase order: an
//    order that depends only on the request's length. Writes the means.
//  * pool_norm_kernel, one workgroup per request: scales the means to unit
//    length (no epsilon, as the reference); thread t adds the squares of
//    columns t, t + 256, ... in order, each with one fmaf.
// A thread's rows are a chain of additions, not of loads: 16 rows' loads are
// issued before the first is added. 3200 rows (a 5000-token request), whose
// chains are 100 rows long: 37.6 us one load at a time on half as many
// workgroups, 11.2 this way, bound by the loads' latency. (Sums of 256-row
// pieces take 5.9, but in another order.)
// ---------------------------------------------------------------------------

__global__ __launch_bounds__(128) void pool_mean_kernel(const uint16_t* __restrict__ norm, Ragged rows, int hidden,
                                                        float* __restrict__ out) {
  __shared__ float part[32][32];
  const int b = blockIdx.y, c0 = blockIdx.x * 32;
  const int r0 = rows.start[b], n = rows.start[b + 1] - r0;
  const int g = threadIdx.x & 3, p = threadIdx.x >> 2;
  const uint16_t* column = norm + (size_t)r0 * hidden + c0 + 8 * g;
  float total[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  // Rows p + at + 32 i of `count` phases' rounds; past the request's end the
  // last row is loaded and zeros are added, which change no sum.
  auto add = [&](int at, auto count) {
    constexpr int kRows = decltype(count)::value;
    half8v v[kRows];
#pragma unroll
    for (int i = 0; i < kRows; ++i) v[i] = *(const half8v*)(column + (size_t)min(p + at + 32 * i, n - 1) * hidden);
    __builtin_amdgcn_sched_barrier(0);  // (the scheduler would take them one at a time, to fit more waves)
#pragma unroll
    for (int i = 0; i < kRows; ++i)
#pragma unroll
      for (int e = 0; e < 8; ++e) total[e] += p + at + 32 * i < n ? (float)v[i][e] : 0.f;
  };
  int at = 0;
  for (; at + 4 * 32 < n; at += 16 * 32) add(at, std::integral_constant<int, 16>{});
  if (at < n) add(at, std::integral_constant<int, 4>{});
#pragma unroll
  for (int e = 0; e < 8; ++e) part[p][8 * g + e] = total[e];
  __syncthreads();
  if (threadIdx.x < 32) {
    float sum = part[0][threadIdx.x];
    for (int q = 1; q < 32; ++q) sum += part[q][threadIdx.x];
    out[(size_t)b * hidden + c0 + threadIdx.x] = sum / (float)n;
  }
}

__global__ __launch_bounds__(256) void pool_norm_kernel(float* __restrict__ out, int hidden) {
  __shared__ float scratch[16];
  float* v = out + (size_t)blockIdx.x * hidden;
  float sq = 0.f;
  float keep[8];  // columns up to 2048 stay in registers
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int c = threadIdx.x + 256 * i;
    keep[i] = c < hidden ? v[c] : 0.f;
  }
#pragma unroll
  for (int i = 0; i < 8; ++i) sq = fmaf(keep[i], keep[i], sq);
  for (int c = threadIdx.x + 2048; c < hidden; c += 256) sq = fmaf(v[c], v[c], sq);
  const float inv = 1.0f / sqrtf(block_sum(sq, scratch));
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int c = threadIdx.x + 256 * i;
    if (c < hidden) v[c] = keep[i] * inv;
  }
  for (int c = threadIdx.x + 2048; c < hidden; c += 256) v[c] *= inv;
}

hipError_t launch_mean_pool(const uint16_t* norm, const Ragged& rows, int hidden, float* out, hipStream_t stream) {
  if (rows.count <= 0) return hipSuccess;
  if (hidden % 64) return hipErrorInvalidValue;
  pool_mean_kernel<<<dim3(hidden / 32, rows.count), 128, 0, stream>>>(norm, rows, hidden, out);
  pool_norm_kernel<<<rows.count, 256, 0, stream>>>(out, hidden);
  return hipGetLastError();
}

}  // namespace nemo
