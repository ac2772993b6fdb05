// dense.hip - the fp32 (non-expert) half of the Qwen3-MoE forward on gfx950:
// the projections, q/k norm, RoPE, causal attention with a KV cache,
// embedding, greedy choice and the vocabulary softmax of
// test_model_trace.c:213-430 and :526-579, bit-identical to the reference.
//
// Every fp32 sum the reference forms is a sequential chain (k ascending,
// each product and sum rounded on its own; the library is compiled with
// -ffp-contract=off).  The kernels keep each chain in one lane and make the
// lanes plentiful: a lane per output row (and token) for the products, a
// lane per score for attention, a lane per head dimension for the weighted V
// sum.  Operands are staged through LDS with coalesced 16-byte loads issued
// a chunk ahead, so that the chain, not the memory, sets the pace (a
// dependent v_add_f32 every ~8 clocks).  Order-free steps (max, expf, the
// products of the softmax) run across lanes.
#include <climits>
#include <cstdlib>
#include <math.h>

#include <mutex>
#include <unordered_map>

#include "dense.h"
#include "moe_device.h"
#include "moe_layer.h"
#include "moe_qtile.h"

namespace moe {
namespace {

__device__ __forceinline__ float4 zero4() { return make_float4(0.0f, 0.0f, 0.0f, 0.0f); }

// acc = (((acc + x0 w0) + x1 w1) + ...) over 4*n4 columns of two LDS rows;
// 16 float4 of each row are read before their 64 dependent adds.
__device__ __forceinline__ float chain_dot(float acc, const float* x, const float* w, int n4) {
  const float4* x4 = reinterpret_cast<const float4*>(x);
  const float4* w4 = reinterpret_cast<const float4*>(w);
  int k4 = 0;
  for (; k4 + 16 <= n4; k4 += 16) {
    float4 xv[16], wv[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) { xv[i] = x4[k4 + i]; wv[i] = w4[k4 + i]; }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const float p0 = xv[i].x * wv[i].x, p1 = xv[i].y * wv[i].y;
      const float p2 = xv[i].z * wv[i].z, p3 = xv[i].w * wv[i].w;
      acc = acc + p0;
      acc = acc + p1;
      acc = acc + p2;
      acc = acc + p3;
    }
  }
  for (; k4 < n4; ++k4) {
    const float4 xv = x4[k4], wv = w4[k4];
    const float p0 = xv.x * wv.x, p1 = xv.y * wv.y, p2 = xv.z * wv.z, p3 = xv.w * wv.w;
    acc = acc + p0;
    acc = acc + p1;
    acc = acc + p2;
    acc = acc + p3;
  }
  return acc;
}

// max(a, b), NaN when either is NaN
__device__ __forceinline__ float nan_max(float a, float b) {
  return (a != a || b != b) ? __builtin_nanf("") : (a > b ? a : b);
}

__device__ __forceinline__ float dense_epilogue(const DenseArgs& a, int m, int n, float acc) {
  float c = acc;
  if (a.bias) c = c + a.bias[n];
  if (a.resid) c = a.resid[(size_t)m * a.ldr + n] + c;
  return c;
}

// ---------------------------------------------------------------- products

// Few tokens (M <= MM = 64 / RW): a block owns RW output rows; wave 0 is the
// consumer, waves 1..NP are producers.  The weight rows and the M token rows
// stream in chunks of KC columns with coalesced 16-byte loads; producer p
// owns chunks p, p + NP, ... and keeps its next chunk in registers, so each
// load has NP chunk-times to arrive (HBM latency, not bandwidth, limits a
// GEMV with this few bytes in flight).  A producer writes its chunk's
// products x[m][k] * w[r][k] into one of NP + 1 LDS buffers; the consumer
// lane m * RW + r sums token m's products with row n0 + r in column order.
// Splitting the roles keeps multiplies and loads out of the chain's wave: a
// pure add chain issues an add every 8 clocks, a chain that also multiplies
// every 12-13 (measured on gfx950).  Columns past K are zero in both
// operands: 0 * 0 = +0 and adding +0 leaves a chain unchanged (a chain that
// starts at +0 and adds round-to-nearest sums is never -0).  Rows past N read
// row N - 1 and are not stored.  K % 4 == 0, 16-byte aligned rows.  Dynamic
// LDS: NP + 1 buffers of M*RW rows of KC + 4 floats, then (NORM) the rows.
//
// NORM: the token rows are staged whole in LDS and rmsnorm'ed first
// (test_model_trace.c:241-255): squares x*x by all threads, their
// sequential sum by the whole block (block_seq_sum), msq / K,
// 1 / sqrtf(msq + eps), then x = (x * inv) * w; the producers' first weight
// chunks load meanwhile.
// Each block also writes a column slice of the normalized rows and
// (PACK = 2 / 3) packs the slice into the activation tables; the last block
// (fused selection) writes the tables' headers.
template <int RW, bool NORM, int PACK, int NP, int MMX = 64 / RW>
__global__ __launch_bounds__(64 * (NP + 1)) void dense_gemv_kernel(DenseArgs a) {
  constexpr int KC = RW >= 16 ? 4096 / RW : 256;
  constexpr int MM = MMX;                    // token rows one block can chain (<= 64 / RW)
  static_assert(MM * RW <= 64, "one consumer lane per chain");
  constexpr int V4 = KC / 4;                 // float4 per row chunk (<= 64)
  constexpr int LD = KC + 4;                 // padded LDS row (floats)
  constexpr int RPL = 64 / V4;               // rows one load instruction covers
  constexpr int NW = RW / RPL;               // W float4 per producer lane per chunk
  constexpr int NB = NP + 1;                 // LDS product buffers
  constexpr int NT = 64 * (NP + 1);
  if constexpr (RW == 1) {   // tokens 16 blockIdx.y .. (17-32 given rows: two groups)
    const int m0 = MM * (int)blockIdx.y;
    a.M = min(a.M - m0, MM);
    a.A += (size_t)m0 * a.lda;
    a.C += (size_t)m0 * a.ldc;
    if (a.resid) a.resid += (size_t)m0 * a.ldr;
    if constexpr (PACK != 0) {
      a.pack_tabs += (size_t)m0 * act_table_bytes(a.K);
      a.pack_part += (size_t)blockIdx.y * gridDim.x * 16 * 2;
    }
  }
  extern __shared__ float4 pl4[];
  float* pl = reinterpret_cast<float*>(pl4);
  __shared__ float inv_s[MM];
  __shared__ int pack_scratch[2];
  __shared__ SeqSumScratch seq;
  __shared__ int ring_full[NP + 1], ring_done;
  if (threadIdx.x <= NP) ring_full[threadIdx.x] = 0;
  if (threadIdx.x == 0) ring_done = 0;
  const int M = a.M, N = a.N, K = a.K;
  const int nc = (K + KC - 1) / KC;
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  const int prod = wave - 1;                 // producer index, -1 for the consumer
  const int n0 = blockIdx.x * RW;
  const int bufsz = M * RW * LD;
  float* xs = pl + NB * bufsz;               // NORM: [M][K] token rows
  const int c4 = lane % V4, r0 = lane / V4;
  float4 rw[NW], rx[MM];
  const float* wsrc[NW];
#pragma unroll
  for (int v = 0; v < NW; ++v)
    wsrc[v] = a.W + (size_t)min(n0 + r0 + v * RPL, N - 1) * a.ldw + 4 * c4;
  auto loadW = [&](int c) {
    const bool in = c * KC + 4 * c4 < K;
#pragma unroll
    for (int v = 0; v < NW; ++v)
      rw[v] = in ? *reinterpret_cast<const float4*>(wsrc[v] + (size_t)c * KC) : zero4();
  };
  auto loadX = [&](int c) {
    const int k = c * KC + 4 * c4;
    const bool in = k < K;
#pragma unroll
    for (int m = 0; m < MM; ++m)
      if (m < M) {
        if constexpr (NORM)
          rx[m] = in ? *reinterpret_cast<const float4*>(xs + (size_t)m * K + k) : zero4();
        else
          rx[m] = in ? *reinterpret_cast<const float4*>(a.A + (size_t)m * a.lda + k) : zero4();
      }
  };
  auto produce = [&](int c) {
    float* P = pl + (c % NB) * bufsz;
#pragma unroll
    for (int m = 0; m < MM; ++m) {
      if (m >= M) break;
#pragma unroll
      for (int v = 0; v < NW; ++v) {
        const float4 w = rw[v], x = rx[m];
        *reinterpret_cast<float4*>(P + (m * RW + r0 + v * RPL) * LD + 4 * c4) =
            make_float4(x.x * w.x, x.y * w.y, x.z * w.z, x.w * w.w);
      }
    }
  };
  if constexpr (NORM) {
    const int k4 = K / 4;
    // The token rows first, alone: issued with the weight chunks of every
    // block they would return behind that burst.  Producer 0 requests chunk
    // 0 once the rows are in (after the staging barrier), so that it arrives
    // while the squares are summed; the other producers' first chunks, needed
    // a chunk-time later, wait until the norm is done.
    constexpr int XR = 2, NWR = 2;
    const bool x_regs = M * k4 <= XR * NT;
    const bool nw_regs = k4 <= NWR * NT;
    float4 xr[XR], nwr[NWR];
#pragma unroll
    for (int u = 0; u < XR; ++u) {
      const int i = (int)threadIdx.x + u * NT;
      xr[u] = (x_regs && i < M * k4)
                  ? *reinterpret_cast<const float4*>(a.A + (size_t)(i / k4) * a.lda + 4 * (i % k4))
                  : zero4();
    }
#pragma unroll
    for (int u = 0; u < NWR; ++u) {
      const int j = (int)threadIdx.x + u * NT;
      nwr[u] = (nw_regs && a.norm_w && j < k4) ? reinterpret_cast<const float4*>(a.norm_w)[j]
                                              : make_float4(1.0f, 1.0f, 1.0f, 1.0f);
    }
    if (x_regs) {
#pragma unroll
      for (int u = 0; u < XR; ++u) {
        const int i = (int)threadIdx.x + u * NT;
        if (i < M * k4) {
          const float4 v = xr[u];
          reinterpret_cast<float4*>(xs)[i] = v;
          reinterpret_cast<float4*>(pl)[i] = make_float4(v.x * v.x, v.y * v.y, v.z * v.z, v.w * v.w);
        }
      }
    } else {
      for (int i = threadIdx.x; i < M * k4; i += NT) {
        const int m = i / k4, j = i % k4;
        const float4 v = *reinterpret_cast<const float4*>(a.A + (size_t)m * a.lda + 4 * j);
        reinterpret_cast<float4*>(xs)[i] = v;
        reinterpret_cast<float4*>(pl)[i] = make_float4(v.x * v.x, v.y * v.y, v.z * v.z, v.w * v.w);
      }
    }
    __syncthreads();
    if (prod == 0 && nc > 0) loadW(0);
    for (int m = 0; m < M; ++m) {
      const float msq = block_seq_sum<NT>(pl + (size_t)m * K, K, seq);
      if (threadIdx.x == 0) inv_s[m] = 1.0f / sqrtf(msq / (float)K + a.eps);
    }
    __syncthreads();
    if (prod > 0 && prod < nc) loadW(prod);
    if (nw_regs) {
      // (a missing weight is 1: the reference multiplies by 1.0f)
#pragma unroll
      for (int u = 0; u < NWR; ++u) {
        const int j = (int)threadIdx.x + u * NT;
        if (j < k4)
          for (int m = 0; m < M; ++m) {
            float4* xp = reinterpret_cast<float4*>(xs + (size_t)m * K) + j;
            const float4 x = *xp, w = nwr[u];
            const float iv = inv_s[m];
            const float v0 = x.x * iv, v1 = x.y * iv, v2 = x.z * iv, v3 = x.w * iv;
            *xp = make_float4(v0 * w.x, v1 * w.y, v2 * w.z, v3 * w.w);
          }
      }
    } else {
      for (int i = threadIdx.x; i < M * K; i += NT) {
        const float v = xs[i] * inv_s[i / K];
        xs[i] = a.norm_w ? v * a.norm_w[i % K] : v * 1.0f;
      }
    }
    __syncthreads();
    // this block's column slice [c0, c1) (a multiple of 8 columns)
    const int sl = ((K + 7) / 8 + (int)gridDim.x - 1) / (int)gridDim.x * 8;
    const int c0 = min(K, (int)blockIdx.x * sl), c1 = min(K, c0 + sl);
    if (a.xn_out)
      for (int m = 0; m < M; ++m)
        for (int i = c0 + threadIdx.x; i < c1; i += NT) a.xn_out[(size_t)m * K + i] = xs[(size_t)m * K + i];
    if constexpr (PACK != 0) {
      const size_t tb = act_table_bytes(K);
      for (int m = 0; m < M; ++m) {
        if (threadIdx.x == 0) { pack_scratch[0] = 1; pack_scratch[1] = 0; }
        __syncthreads();
        int nl;
        uint32_t sum;
        pack_act_cols<PACK == 3>(xs + (size_t)m * K, K, c0, c1, a.pack_tabs + m * tb, threadIdx.x, NT,
                                 nl, sum);
        // wave reductions, then one LDS atomic per wave
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
          const int on = __shfl_xor(nl, off, kWave);
          nl = on > nl ? on : nl;
          sum += (uint32_t)__shfl_xor((int)sum, off, kWave);
        }
        if (lane == 0) {
          atomicMax(&pack_scratch[0], nl);
          atomicAdd(reinterpret_cast<unsigned*>(&pack_scratch[1]), sum);
        }
        __syncthreads();
        if (threadIdx.x == 0) {
          uint32_t* pp = a.pack_part + ((size_t)m * gridDim.x + blockIdx.x) * 2;
          pp[0] = (uint32_t)pack_scratch[0];
          pp[1] = (uint32_t)pack_scratch[1];
        }
      }
    }
  }
  if constexpr (!NORM) {
    if (prod >= 0 && prod < nc) loadW(prod);
    if constexpr (PACK != 0) {
      // up to 16 given rows: this block's column slice [c0, c1) of each
      // token row into its activation table, V columns a thread, while the
      // first chunks load; the slice's partial header {limbs, sum} goes to
      // pack_part[block][token] (select_kernel writes the headers)
      static_assert(MM <= 16, "partial headers of up to 16 tokens a block");
      constexpr int V = PACK == 3 ? 8 : 4;
      __shared__ unsigned pk[16][2];
      if (threadIdx.x < 16) { pk[threadIdx.x][0] = 1u; pk[threadIdx.x][1] = 0u; }
      __syncthreads();
      const int sl = ((K + 7) / 8 + (int)gridDim.x - 1) / (int)gridDim.x * 8;
      const int c0 = min(K, (int)blockIdx.x * sl), c1 = min(K, c0 + sl);
      const int G = (c1 - c0 + V - 1) / V;
      const size_t tb = act_table_bytes(K);
      for (int i = threadIdx.x; i < M * G; i += NT) {
        const int m = i / G, g0 = c0 + (i % G) * V;
        int nl;
        uint32_t sum;
        pack_act_cols<PACK == 3>(a.A + (size_t)m * a.lda, K, g0, min(c1, g0 + V), a.pack_tabs + m * tb, 0, 1,
                                 nl, sum);
        atomicMax(&pk[m][0], (unsigned)nl);
        atomicAdd(&pk[m][1], sum);
      }
      __syncthreads();
      if (threadIdx.x < M)
        reinterpret_cast<uint2*>(a.pack_part)[(size_t)blockIdx.x * 16 + threadIdx.x] =
            make_uint2(pk[threadIdx.x][0], pk[threadIdx.x][1]);
    }
  }
  // The ring's hand-over: a producer stores k + 1 into ring_full[k % NB]
  // after writing chunk k, the consumer the number of chunks it has summed
  // into ring_done; a producer waits for ring_done >= k - NB + 1 before
  // reusing a buffer, the consumer for ring_full[c % NB] >= c + 1.  Neither
  // side waits on itself, so every wait ends.
  __syncthreads();   // the ring counters are zero
  if (prod >= 0) {
    if (prod < nc) loadX(prod);
    for (int k = prod; k < nc; k += NP) {
      if (k >= NB) ring_wait(&ring_done, k - NB + 1, true);
      produce(k);
      ring_post(&ring_full[k % NB], k + 1);
      if (k + NP < nc) {
        loadW(k + NP);
        loadX(k + NP);
      }
    }
  } else {
    const int m = lane / RW, r = lane % RW;
    const bool live = m < M;
    float acc = 0.0f;
    for (int c = 0; c < nc; ++c) {
      ring_wait(&ring_full[c % NB], c + 1, false);
      if (live) acc = chain_sum(acc, pl + (c % NB) * bufsz + lane * LD, V4);
      ring_post(&ring_done, c + 1);
    }
    const int n = n0 + r;
    float c = -__builtin_inff();
    if (live && n < N) {
      c = dense_epilogue(a, m, n, acc);
      a.C[(size_t)m * a.ldc + n] = c;
    }
    if (a.amax_part) {   // M == 1: the block's largest output, NaN if any is NaN
      float v = c;
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) v = nan_max(v, __shfl_xor(v, off, kWave));
      if (lane == 0) a.amax_part[blockIdx.x] = v;
    }
  }
  if constexpr (RW == 16) {
    if (a.sel_counter) {
      // the last block to finish selects the experts of every token (and
      // writes the activation tables' headers from the slices' partials)
      __shared__ int last;
      __shared__ int sidx[NP + 1][kMaxTopK];
      __shared__ float sval[NP + 1][kMaxTopK], sexp[NP + 1][kMaxTopK];
      __threadfence();
      __syncthreads();
      if (threadIdx.x == 0) {
        const unsigned prev = atomicAdd(a.sel_counter, 1u);
        last = prev == gridDim.x - 1;
        if (last) *a.sel_counter = 0u;
      }
      __syncthreads();
      if (last) {
        __threadfence();
        if constexpr (PACK != 0) {
          if (threadIdx.x < M) {
            const int m = threadIdx.x;
            uint32_t nl = 1, sum = 0;
            for (unsigned b = 0; b < gridDim.x; ++b) {
              const uint32_t* pp = a.pack_part + ((size_t)m * gridDim.x + b) * 2;
              nl = pp[0] > nl ? pp[0] : nl;
              sum += pp[1];
            }
            uint32_t* hh = reinterpret_cast<uint32_t*>(a.pack_tabs + m * act_table_bytes(K));
            hh[0] = nl;
            hh[1] = sum;
          }
        }
        // one wave per token; keys in the product buffers (free now)
        uint64_t* keys = reinterpret_cast<uint64_t*>(pl) + (size_t)wave * 1024;
        for (int m = wave; m < M; m += NP + 1) {
          const size_t o = (size_t)m * a.sel_topk;
          select_token_any(a.C + (size_t)m * a.ldc, N, a.sel_topk, keys, sidx[wave], sval[wave],
                           sexp[wave], a.sel_idx + o, a.sel_p + o,
                           a.sel_idx_user ? a.sel_idx_user + o : nullptr,
                           a.sel_p_user ? a.sel_p_user + o : nullptr);
        }
      }
    }
  }
}

// Few tokens, few rows (the router): one block per (output row, token); with
// NORM one token.  The token row is staged in LDS (normalized first
// when NORM, the sum of squares by block_seq_sum), the products x[k] *
// W[n][k] are formed into LDS and summed in order by block_seq_sum, so a row
// costs about K / 8 dependent adds instead of K.  With PACK each block packs its column slice of its
// token's (normalized) row into that token's activation table (row_finish_kernel writes the
// header and, with a fused selection, picks the experts).
// 512 threads: two waves per SIMD.  A wave issues a VALU instruction about
// every 8 clocks whether or not it depends on the previous one, so the
// candidate chains of block_seq_sum fill a SIMD only with two waves on it.
constexpr int kRowThreads = 512;
constexpr int kRowMaxK = 8192;

template <bool NORM, int PACK>
__global__ __launch_bounds__(kRowThreads) void dense_row_kernel(DenseArgs a) {
  extern __shared__ float4 rl4[];
  const int K = a.K, k4 = K / 4, n = blockIdx.x, m = blockIdx.y;
  float* xs = reinterpret_cast<float*>(rl4);   // [K] the token row
  float* pv = xs + K;                          // [K] squares, then products, then keys
  float4* xs4 = rl4;
  float4* pv4 = rl4 + k4;
  __shared__ SeqSumScratch seq;
  __shared__ int pack_scratch[2];
  __shared__ float inv_s;
  const int tid = threadIdx.x, lane = tid % kWave;
  if (a.epoch_bump && n == 0 && m == 0 && tid == 0) {
    const uint32_t e = *a.epoch_bump + 1u;
    *a.epoch_bump = e ? e : 1u;
  }
  constexpr int WV = kRowMaxK / 4 / kRowThreads;
  // the token row (and norm weights) into registers first, then the weight
  // row (a wave's loads complete in order: the LDS staging waits only for
  // the token row)
  const float4* x4 = reinterpret_cast<const float4*>(a.A + (size_t)m * a.lda);
  const float4* nw4g = reinterpret_cast<const float4*>(a.norm_w);
  float4 xv[WV], nv[WV];
#pragma unroll
  for (int u = 0; u < WV; ++u) {
    const int i = tid + kRowThreads * u;
    xv[u] = i < k4 ? x4[i] : zero4();
    nv[u] = (NORM && a.norm_w && i < k4) ? nw4g[i] : make_float4(1.0f, 1.0f, 1.0f, 1.0f);
  }
  const float4* wr = reinterpret_cast<const float4*>(a.W + (size_t)n * a.ldw);
  float4 w[WV];
#pragma unroll
  for (int u = 0; u < WV; ++u) {
    const int i = tid + kRowThreads * u;
    w[u] = i < k4 ? wr[i] : zero4();
  }
#pragma unroll
  for (int u = 0; u < WV; ++u) {
    const int i = tid + kRowThreads * u;
    if (i < k4) {
      const float4 v = xv[u];
      xs4[i] = v;
      if (NORM) pv4[i] = make_float4(v.x * v.x, v.y * v.y, v.z * v.z, v.w * v.w);
    }
  }
  __syncthreads();
  if constexpr (NORM) {
    const float msq = block_seq_sum<kRowThreads>(pv, K, seq);
    if (tid == 0) inv_s = 1.0f / sqrtf(msq / (float)K + a.eps);
    __syncthreads();
    // (a missing weight is 1: the reference multiplies by 1.0f)
    const float iv = inv_s;
#pragma unroll
    for (int u = 0; u < WV; ++u) {
      const int i = tid + kRowThreads * u;
      if (i < k4) {
        const float4 x = xv[u], g = nv[u];
        const float v0 = x.x * iv, v1 = x.y * iv, v2 = x.z * iv, v3 = x.w * iv;
        xs4[i] = make_float4(v0 * g.x, v1 * g.y, v2 * g.z, v3 * g.w);
      }
    }
    __syncthreads();
  }
  // this block's column slice [c0, c1) (a multiple of 8 columns) of the
  // (normalized) row: to xn_out, and packed into the x tables' planes
  const int sl = ((K + 7) / 8 + (int)gridDim.x - 1) / (int)gridDim.x * 8;
  const int c0 = min(K, (int)blockIdx.x * sl), c1 = min(K, c0 + sl);
  if (NORM && a.xn_out)
    for (int i = c0 + tid; i < c1; i += kRowThreads) a.xn_out[i] = xs[i];
  if constexpr (PACK != 0) {
    if (tid == 0) { pack_scratch[0] = 1; pack_scratch[1] = 0; }
    __syncthreads();
    int nl;
    uint32_t sum;
    pack_act_cols<PACK == 3>(xs, K, c0, c1, a.pack_tabs + (size_t)m * act_table_bytes(K), tid, kRowThreads,
                             nl, sum);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const int on = __shfl_xor(nl, off, kWave);
      nl = on > nl ? on : nl;
      sum += (uint32_t)__shfl_xor((int)sum, off, kWave);
    }
    if (lane == 0) {
      atomicMax(&pack_scratch[0], nl);
      atomicAdd(reinterpret_cast<unsigned*>(&pack_scratch[1]), sum);
    }
    __syncthreads();
    if (tid == 0) {
      uint32_t* pp = a.pack_part + ((size_t)m * gridDim.x + blockIdx.x) * 2;
      pp[0] = (uint32_t)pack_scratch[0];
      pp[1] = (uint32_t)pack_scratch[1];
    }
  }
  // products x[k] * W[n][k], then their sum in column order
#pragma unroll
  for (int u = 0; u < WV; ++u) {
    const int i = tid + kRowThreads * u;
    if (i < k4) {
      const float4 x = xs4[i];
      pv4[i] = make_float4(x.x * w[u].x, x.y * w[u].y, x.z * w[u].z, x.w * w[u].w);
    }
  }
  __syncthreads();
  const float acc = block_seq_sum<kRowThreads>(pv, K, seq);
  if (tid == 0) a.C[(size_t)m * a.ldc + n] = dense_epilogue(a, m, n, acc);
}

// 5-16 tokens, few rows: a block per (output row, four tokens), its 512
// threads four groups of 128 side by side, each the row kernel on its own
// token -- products x[k] * W[n][k] into its LDS slice, summed in order by
// group_seq_sum (four candidate chains per thread).  No norm.  With PACK
// each group also packs the block's column slice of its token's row into
// the token's activation table and leaves the slice's partial header at
// pack_part[slice][token] (uint2 {limbs, sum}; select_kernel combines them).
constexpr int kRowGroups = 4;
constexpr int kRowGroupThreads = kRowThreads / kRowGroups;
constexpr int kRowsMaxK = 4096;

template <int PACK>
__global__ __launch_bounds__(kRowThreads) void dense_rows4_kernel(DenseArgs a) {
  extern __shared__ float4 rg4[];   // [kRowGroups][K] products
  __shared__ SeqSumScratch seq[kRowGroups];
  __shared__ int pk[kRowGroups][2];
  const int K = a.K, k4 = K / 4, n = blockIdx.x;
  const int g = threadIdx.x / kRowGroupThreads, gt = threadIdx.x % kRowGroupThreads;
  const int mg = blockIdx.y * kRowGroups + g;   // this group's token (past M: a repeat, not written)
  const int m = min(mg, a.M - 1);
  float4* pv4 = rg4 + (size_t)g * k4;
  const float4* x4 = reinterpret_cast<const float4*>(a.A + (size_t)m * a.lda);
  const float4* w4 = reinterpret_cast<const float4*>(a.W + (size_t)n * a.ldw);
  constexpr int WV = kRowsMaxK / 4 / kRowGroupThreads;
  float4 xv[WV], wv[WV];
#pragma unroll
  for (int u = 0; u < WV; ++u) {
    const int i = gt + kRowGroupThreads * u;
    xv[u] = i < k4 ? x4[i] : zero4();
  }
#pragma unroll
  for (int u = 0; u < WV; ++u) {
    const int i = gt + kRowGroupThreads * u;
    wv[u] = i < k4 ? w4[i] : zero4();
  }
  if constexpr (PACK != 0) {
    // the block's column slice [c0, c1) (a multiple of 8 columns)
    const int sl = ((K + 7) / 8 + (int)gridDim.x - 1) / (int)gridDim.x * 8;
    const int c0 = min(K, (int)blockIdx.x * sl), c1 = min(K, c0 + sl);
    if (gt == 0) { pk[g][0] = 1; pk[g][1] = 0; }
    int nl = 1;
    uint32_t sum = 0;
    if (mg < a.M)
      pack_act_cols<PACK == 3>(a.A + (size_t)m * a.lda, K, c0, c1, a.pack_tabs + (size_t)m * act_table_bytes(K),
                               gt, kRowGroupThreads, nl, sum);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const int on = __shfl_xor(nl, off, kWave);
      nl = on > nl ? on : nl;
      sum += (uint32_t)__shfl_xor((int)sum, off, kWave);
    }
    __syncthreads();
    if (threadIdx.x % kWave == 0) {
      atomicMax(&pk[g][0], nl);
      atomicAdd(reinterpret_cast<unsigned*>(&pk[g][1]), sum);
    }
  }
#pragma unroll
  for (int u = 0; u < WV; ++u) {
    const int i = gt + kRowGroupThreads * u;
    if (i < k4)
      pv4[i] = make_float4(xv[u].x * wv[u].x, xv[u].y * wv[u].y, xv[u].z * wv[u].z, xv[u].w * wv[u].w);
  }
  __syncthreads();
  if constexpr (PACK != 0) {
    if (gt == 0 && mg < a.M)
      reinterpret_cast<uint2*>(a.pack_part)[(size_t)n * 16 + mg] = make_uint2((unsigned)pk[g][0], (unsigned)pk[g][1]);
  }
  const float acc = group_seq_sum<kRowGroupThreads>(reinterpret_cast<const float*>(pv4), K, seq[g], gt);
  if (gt == 0 && mg < a.M) a.C[(size_t)m * a.ldc + n] = dense_epilogue(a, m, n, acc);
}

// After dense_row_kernel (a kernel boundary instead of a fence in each of
// its blocks): each token's activation-table header from its slices'
// partials and its expert selection, one wave per token (M <= 4).
constexpr int kRowFinishWaves = 4;
__global__ __launch_bounds__(kRowFinishWaves * kWave) void row_finish_kernel(DenseArgs a) {
  __shared__ uint64_t keys[kRowFinishWaves][1024];
  __shared__ int sidx[kRowFinishWaves][kMaxTopK];
  __shared__ float sval[kRowFinishWaves][kMaxTopK], sexp[kRowFinishWaves][kMaxTopK];
  const int lane = threadIdx.x % kWave, m = threadIdx.x / kWave;
  if (a.pack_dtype && m < a.M) {
    uint32_t nl = 1, sum = 0;
    for (int b = lane; b < a.N; b += kWave) {
      const uint32_t* pp = a.pack_part + ((size_t)m * a.N + b) * 2;
      nl = pp[0] > nl ? pp[0] : nl;
      sum += pp[1];
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const uint32_t on = (uint32_t)__shfl_xor((int)nl, off, kWave);
      nl = on > nl ? on : nl;
      sum += (uint32_t)__shfl_xor((int)sum, off, kWave);
    }
    if (lane == 0) {
      uint32_t* hh = reinterpret_cast<uint32_t*>(a.pack_tabs + (size_t)m * act_table_bytes(a.K));
      hh[0] = nl;
      hh[1] = sum;
    }
  }
  if (m >= a.M) return;
  const size_t o = (size_t)m * a.sel_topk;
  select_token_any(a.C + (size_t)m * a.ldc, a.N, a.sel_topk, keys[m], sidx[m], sval[m], sexp[m],
                   a.sel_idx + o, a.sel_p + o, a.sel_idx_user ? a.sel_idx_user + o : nullptr,
                   a.sel_p_user ? a.sel_p_user + o : nullptr);
}

// Many tokens, products on the matrix cores: v_mfma_f32_16x16x1_4b with C =
// 0 and one column per block is four 16 x 16 outer products whose every
// element is one product x w rounded once, bit for bit v_mul_f32's (checked
// over random bit patterns, products in and below the denormal range and
// infinities), so only the adds of the chains are left to the VALU.
// A wave owns 16 tokens x NB tiles of 16 rows, a block of four waves 16 WX
// tokens x 16 NB (4 / WX) rows; a lane holds 4 NB chains (tokens 4 (lane /
// 16) + r, row lane % 16 of each tile).  The four blocks of one MFMA are four
// columns of one tile: lane (b, i) = (lane / 16, lane % 16) feeds token i and
// row i of column 4b + c in MFMA c, and result register 4b + r of MFMA c is
// the product of that column, so the 16 products of a chain's 16 columns are
// registers of its own lane.  One ds_read_b128 a lane feeds four MFMAs.
// Operands stream through a D-buffer LDS ring of KC-column chunks with
// global_load_lds_dwordx4, XOR-swizzled, one barrier a chunk.
//
// Bound: VALU issue.  fp32 MFMA and VALU share the fp32 units (a loop of both
// takes the sum of their times): 2.05 clocks per 64 products and ~2.3 per 64
// adds with four waves a SIMD, against 4.9 for v_mul_f32 + v_add_f32 whose
// operand reads also bind on LDS.  Four MFMAs, then their 64 adds: switching
// between the two costs clocks (4.2 per 64 products in this order, 5.0 with an
// MFMA before every 16 adds; 6.6 with one wave a SIMD).  512 x 5120 x 2048
// (the Q/K/V product of a 512-token prompt): 232 -> 172 us; 512 x 2048 x 4096
// (its O product): 190 -> 156; 100 x 2048 x 4096: 181 -> 60; the add and
// product floor of the first is 148.
typedef float v16f __attribute__((ext_vector_type(16)));

// The products of 16 columns of a 16 x 16 tile (x, w: the lane's columns 4b ..
// 4b + 3 of its token and row): p[c][4b + r] belongs to column 4b + c, chain r.
__device__ __forceinline__ void mfma_products(const float4& x, const float4& w, v16f (&p)[4]) {
  p[0] = __builtin_amdgcn_mfma_f32_16x16x1f32(x.x, w.x, v16f{}, 0, 0, 0);
  p[1] = __builtin_amdgcn_mfma_f32_16x16x1f32(x.y, w.y, v16f{}, 0, 0, 0);
  p[2] = __builtin_amdgcn_mfma_f32_16x16x1f32(x.z, w.z, v16f{}, 0, 0, 0);
  p[3] = __builtin_amdgcn_mfma_f32_16x16x1f32(x.w, w.w, v16f{}, 0, 0, 0);
}

__device__ __align__(16) const float kDenseZero[4] = {};

typedef float f32x4_any __attribute__((ext_vector_type(4), aligned(4)));

// ANY: rows of any length at any 4-byte alignment, which the direct loads to
// LDS do not take: each lane's 16 bytes of the next chunk go through registers
// while the chunk before is multiplied (two LDS buffers).  Against a thread an
// output (dense_generic_kernel, bound by its uncoalesced row reads): 1 x 8192 x
// 4095 1822 -> 64 us, 7 x 3000 x 1001 288 -> 18, 100 x 2048 x 4095 1522 -> 64,
// 512 x 5120 x 2047 20.9 ms -> 179 us (the direct loads at K = 2048: 170).  The
// two large tiles spill at four waves a SIMD: 247 us there, 179 at three.
template <int WX, int NB, int KC, int D, bool ANY>
__global__ __launch_bounds__(256, ANY && NB >= 4 ? 3 : 4) void dense_mfma_kernel(DenseArgs a) {
  constexpr int WN = 4 / WX;
  constexpr int RX = 16 * WX, RW = 16 * NB * WN, R = RX + RW;
  constexpr int SL = KC / 4;                 // 16-byte slots of an LDS row
  constexpr int RPI = 64 / SL;               // rows one load instruction covers
  constexpr int NI = R / RPI;                // load instructions of a chunk
  constexpr int NL = (NI + 3) / 4;           // per wave
  static_assert(R % RPI == 0, "whole load instructions");
  __shared__ float4 lds4[D][R * SL];
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int b = lane / 16, j = lane % 16;
  const int wx = wave % WX, wn = wave / WX;
  const int t0 = blockIdx.y * RX, n0 = blockIdx.x * RW;
  const int nc = (a.K + KC - 1) / KC;
  // slot s of row r sits at s ^ sw(r): the 16 lanes of one read (rows j, one
  // slot) then cover all 64 banks
  auto sw = [](int r) { return KC == 64 ? r & 15 : (r >> 1) & 7; };
  const float* src[NL];
  int col[NL];
#pragma unroll
  for (int v = 0; v < NL; ++v) {
    const int row = RPI * ((wave + 4 * v) % NI) + lane / SL;   // past the tile: another wave's rows again
    col[v] = 4 * ((lane % SL) ^ sw(row));
    src[v] = row < RX ? a.A + (size_t)min(t0 + row, a.M - 1) * a.lda + (ANY ? 0 : col[v])
                      : a.W + (size_t)min(n0 + row - RX, a.N - 1) * a.ldw + (ANY ? 0 : col[v]);
  }
  f32x4_any next[ANY ? NL : 1];
  // K >= 4: a load that would pass the row's end is moved back to end with it,
  // and its columns moved down (zeros from K on) on the way to LDS
  auto fetch = [&](int c) {
#pragma unroll
    for (int v = 0; v < NL; ++v)
      next[v] = *reinterpret_cast<const f32x4_any*>(src[v] + min(c * KC + col[v], a.K - 4));
  };
  auto store = [&](int c, int h) {
    if ((c + 1) * KC > a.K) {
#pragma unroll
      for (int v = 0; v < NL; ++v) {
        const int d = c * KC + col[v] - min(c * KC + col[v], a.K - 4);
        if (d & 1) next[v] = f32x4_any{next[v][1], next[v][2], next[v][3], 0.0f};
        if (d & 2) next[v] = f32x4_any{next[v][2], next[v][3], 0.0f, 0.0f};
        if (d >= 4) next[v] = f32x4_any{0.0f, 0.0f, 0.0f, 0.0f};
      }
    }
#pragma unroll
    for (int v = 0; v < NL; ++v)
      lds4[h][((wave + 4 * v) % NI) * 64 + lane] = make_float4(next[v][0], next[v][1], next[v][2], next[v][3]);
  };
  auto load = [&](int c, int h) {
    uint8_t* l = reinterpret_cast<uint8_t*>(lds4[h]);
    if ((c + 1) * KC <= a.K) {
#pragma unroll
      for (int v = 0; v < NL; ++v)
        lds_load16(src[v] + (size_t)c * KC, l + ((wave + 4 * v) % NI) * 1024);
    } else {
#pragma unroll
      for (int v = 0; v < NL; ++v)
        lds_load16(c * KC + col[v] < a.K ? src[v] + (size_t)c * KC : kDenseZero,
                   l + ((wave + 4 * v) % NI) * 1024);
    }
  };
  float acc[NB][4];
#pragma unroll
  for (int t = 0; t < NB; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[t][r] = 0.0f;
  static_assert(!ANY || D == 2, "the register path alternates two buffers");
  if constexpr (ANY) {
    fetch(0);
    store(0, 0);
  } else {
    for (int p = 0; p < D - 1; ++p) load(min(p, nc - 1), p);
  }
#pragma unroll 1
  for (int c = 0; c < nc; ++c) {
    if constexpr (ANY) {
      __syncthreads();   // chunk c is in LDS, every wave is done with chunk c - 1
      fetch(min(c + 1, nc - 1));
    } else {
      stage_sync<(D - 2) * NL>();
      load(min(c + D - 1, nc - 1), (c + D - 1) % D);
    }
    const float4* B = lds4[c % D] + j * SL;
    constexpr int STEPS = KC / 16 * NB;   // 16 columns of one row tile each
    auto read_x = [&](int g) { return B[16 * wx * SL + ((4 * g + b) ^ sw(j))]; };
    auto read_w = [&](int t, int g) { return B[(RX + 16 * (NB * wn + t)) * SL + ((4 * g + b) ^ sw(j))]; };
    float4 x = read_x(0), w = read_w(0, 0);
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      const int t = i % NB;
      float4 xn = x, wn4 = w;
      if (i + 1 < STEPS) {
        wn4 = read_w((i + 1) % NB, (i + 1) / NB);
        if ((i + 1) % NB == 0) xn = read_x((i + 1) / NB);
      }
      asm volatile("" ::: "memory");   // the next step's operands are requested here, not sunk to their use
      v16f p[4];
      mfma_products(x, w, p);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < 16; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[t][r] = acc[t][r] + p[k % 4][4 * (k / 4) + r];
      if constexpr (ANY)   // the adds stay here, not sunk towards the store
        asm volatile("" : "+v"(acc[t][0]), "+v"(acc[t][1]), "+v"(acc[t][2]), "+v"(acc[t][3]));
      __builtin_amdgcn_sched_barrier(0);
      x = xn;
      w = wn4;
    }
    if constexpr (ANY) {
      store(min(c + 1, nc - 1), (c + 1) % D);
    }
  }
  if constexpr (!ANY) stage_sync<0>();   // the clamped loads past the last chunk have landed
#pragma unroll
  for (int t = 0; t < NB; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int tok = t0 + 16 * wx + 4 * b + r, n = n0 + 16 * (NB * wn + t) + j;
      if (tok < a.M && n < a.N) a.C[(size_t)tok * a.ldc + n] = dense_epilogue(a, tok, n, acc[t][r]);
    }
}

// Any shape or alignment: one thread per output, plain loads (unaligned rows
// of a few columns, more rows than a grid of tiles takes).
__global__ __launch_bounds__(256) void dense_generic_kernel(DenseArgs a) {
  const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
  if (i >= (long long)a.M * a.N) return;
  const int m = (int)(i / a.N), n = (int)(i % a.N);
  const float* x = a.A + (size_t)m * a.lda;
  const float* w = a.W + (size_t)n * a.ldw;
  float acc = 0.0f;
  for (int k = 0; k < a.K; ++k) {
    const float p = x[k] * w[k];
    acc = acc + p;
  }
  a.C[(size_t)m * a.ldc + n] = dense_epilogue(a, m, n, acc);
}

// ---------------------------------------------------------------- heads

constexpr int kMaxHd = 512;

// Up to two head rows (v0 and, if v1, v1; LDS, hd values each) through the
// per-head RMSNorm of test_model_trace.c:381-402 (when the weight is given:
// squares by all lanes, the sequential sum in lane 0 (row 0) and lane 1
// (row 1) side by side, inv = 1/sqrtf(msq/hd + eps), v = (v*inv)*w) and
// RoPE (:326-336: the pair (i, i + hd/2) turned by cos/sin of the row's
// position, each product rounded, then one subtraction / addition) into
// out0 / out1 (global or LDS).  Everything the rows need (weights, cos/sin)
// is read from LDS or registers, so no global load sits between the steps.
// Called by all 64 threads of a one-wave block; sq: LDS scratch [2][hd].
__device__ void heads_prep(float* v0, float* v1, const float* w0, const float* w1, float eps,
                           int hd, const float* cs, const float* sn, float* sq, float* inv_s,
                           float* out0, float* out1) {
  const int lane = threadIdx.x, d2 = hd / 2;
  const bool n0 = w0 != nullptr, n1 = v1 && w1;
  if (n0 || n1) {
    for (int d = lane; d < hd; d += 64) {
      if (n0) sq[d] = v0[d] * v0[d];
      if (n1) sq[hd + d] = v1[d] * v1[d];
    }
    __syncthreads();
    if ((lane == 0 && n0) || (lane == 1 && n1)) {
      const float msq = chain_sum(0.0f, sq + lane * hd, hd / 4);
      const float mean = msq / (float)hd;
      inv_s[lane] = 1.0f / sqrtf(mean + eps);
    }
    __syncthreads();
    for (int d = lane; d < hd; d += 64) {
      if (n0) {
        const float s = v0[d] * inv_s[0];
        v0[d] = s * w0[d];
      }
      if (n1) {
        const float s = v1[d] * inv_s[1];
        v1[d] = s * w1[d];
      }
    }
    __syncthreads();
  }
  for (int i = lane; i < d2; i += 64) {
    const float c = cs[i], s = sn[i];
    {
      const float e = v0[i], o = v0[i + d2];
      const float ec = e * c, os = o * s, oc = o * c, es = e * s;
      out0[i] = ec - os;
      out0[i + d2] = oc + es;
    }
    if (v1) {
      const float e = v1[i], o = v1[i + d2];
      const float ec = e * c, os = o * s, oc = o * c, es = e * s;
      out1[i] = ec - os;
      out1[i + d2] = oc + es;
    }
  }
}

// 4 RW consecutive (token, head) rows of [Q | K | V] a block (row q is head q %
// (nq + 2 nkv) of token q / (nq + 2 nkv), hd wide): q/k rows through the
// per-head RMSNorm and RoPE of heads_prep at position pos0 + t (Q in place, K
// to the cache), V rows to the cache unchanged.  Latency: one lane a row runs
// its sequential sum of squares, the rows of a block side by side.  RW = 4 once
// its blocks fill the chip: one row a block left it waiting on 20,480 such
// chains (512 tokens, 40 heads of 128, 18.1 -> 8.4 us); RW = 1 below, where
// more rows a block only add to the wait (3 tokens 6.1 -> 4.7 us, 40 tokens
// 5.5 -> 4.8).
template <int RW>
__global__ __launch_bounds__(256, RW == 4 ? 5 : 1) void heads_kernel(HeadArgs a) {
  constexpr int NR = 4 * RW;
  extern __shared__ float hrow[];   // [NR][hd + 4] rows, then the same of squares
  __shared__ float inv_s[NR];
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int hd = a.hd, d2 = hd / 2, LD = hd + 4, H = a.nq + 2 * a.nkv;
  const long long q0 = (long long)blockIdx.x * NR, nrow = (long long)a.T * H;
  float* sq = hrow + NR * LD;
  float* row[RW];
  int t[RW], h[RW];
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    const long long q = min(q0 + wave * RW + i, nrow - 1);
    t[i] = (int)(q / H);
    h[i] = (int)(q % H);
    row[i] = a.qkv + (size_t)t[i] * a.ld + (size_t)h[i] * hd;
  }
  for (int d = lane; d < hd; d += kWave) {
    float v[RW];
#pragma unroll
    for (int i = 0; i < RW; ++i) v[i] = row[i][d];
#pragma unroll
    for (int i = 0; i < RW; ++i) {
      hrow[(wave * RW + i) * LD + d] = v[i];
      sq[(wave * RW + i) * LD + d] = v[i] * v[i];
    }
  }
  // weights, cosine and sine of a lane's pair of columns; the first pair's
  // are requested here (RW = 1: four rows' would cost a block its neighbour,
  // 512 tokens 8.4 -> 10.1 us)
  struct Pair { float w0, w1, c, s; };
  auto fetch = [&](int i, int d) {
    const float* w = h[i] < a.nq ? a.q_norm : a.k_norm;
    const size_t at = (size_t)(a.pos0 + t[i]) * d2 + d;
    return Pair{w ? w[d] : 1.0f, w ? w[d + d2] : 1.0f, a.rope_cos[at], a.rope_sin[at]};
  };
  Pair first{};
  if (RW == 1 && lane < d2) first = fetch(0, lane);
  __syncthreads();
  if ((int)threadIdx.x < NR) {
    const float msq = chain_sum(0.0f, sq + threadIdx.x * LD, hd / 4);
    inv_s[threadIdx.x] = 1.0f / sqrtf(msq / (float)hd + a.eps);
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < RW; ++i) {
    if (q0 + wave * RW + i >= nrow) break;
    const int pos = a.pos0 + t[i];
    const float* v = hrow + (wave * RW + i) * LD;
    if (h[i] >= a.nq + a.nkv) {
      float* dst = a.vc + ((size_t)(h[i] - a.nq - a.nkv) * a.max_seq + pos) * hd;
      for (int d = lane; d < hd; d += kWave) dst[d] = v[d];
      continue;
    }
    const bool normed = (h[i] < a.nq ? a.q_norm : a.k_norm) != nullptr;
    float* out = h[i] < a.nq ? row[i] : a.kc + ((size_t)(h[i] - a.nq) * a.max_seq + pos) * hd;
    const float inv = inv_s[wave * RW + i];
    for (int d = lane; d < d2; d += kWave) {
      const Pair p = RW == 1 && d == lane ? first : fetch(i, d);
      float e = v[d], o = v[d + d2];
      if (normed) {
        e = e * inv;
        o = o * inv;
        e = e * p.w0;
        o = o * p.w1;
      }
      const float ec = e * p.c, os = o * p.s, oc = o * p.c, es = e * p.s;
      out[d] = ec - os;
      out[d + d2] = oc + es;
    }
  }
}

// ---------------------------------------------------------------- attention

// Scores of query row t, head h against cache positions tk0 .. tk0 + 63
// (<= pos0 + t): lane i runs the chain dot = (((0 + q0 k0) + q1 k1) + ...)
// over hd for position tk0 + i and stores dot * scale.  REG (hd <= 128):
// each lane loads its K row straight into registers (one round trip);
// otherwise the 64 K rows are staged in LDS.  fuse_heads (T == 1, position
// P = pos0): q is normed and rotated here; the block holding position P
// computes K's row P the same way (the cache does not have it yet) and, for
// the first query head of each KV group, writes K and V row P into the
// caches.  All global loads are issued first.
constexpr int kRegHd = 128;

// (x, y) work indices of this block in a 2-D grid, permuted so that blocks
// with consecutive y (heads of one KV group) share an XCD: blocks are dealt
// to the 8 XCDs in turn, so XCD k runs the blocks whose linear index is k
// mod 8, and those get logical indices k n/8 .. k n/8 + n/8 - 1 (x fastest).
// The K and V rows a KV head's blocks read then come from one XCD's L2
// instead of every XCD's.  The identity when n is not a multiple of 8 or
// with MOEHIP_ATTN_NO_XCD set.
__device__ __forceinline__ void attn_xcd_map(bool on, int* bx, int* by) {
  const int gx = (int)gridDim.x, n = gx * (int)gridDim.y;
  const int L = (int)blockIdx.x + gx * (int)blockIdx.y;
  if (!on || n % 8) {
    *bx = (int)blockIdx.x;
    *by = (int)blockIdx.y;
    return;
  }
  const int Lg = (L % 8) * (n / 8) + L / 8;
  *bx = Lg % gx;
  *by = Lg / gx;
}

template <bool REG>
__global__ __launch_bounds__(64) void attn_scores_kernel(AttnArgs a) {
  extern __shared__ float lds[];
  const int hd = a.hd, LD = hd + 4, d2 = hd / 2;
  const int hdp = (hd + 3) & ~3;
  float* q = lds;                       // [hd] the query (rotated)
  float* kt = q + hdp;                  // REG: [hd] K row P; else [64][LD] K rows
  float* qraw = kt + (REG ? hdp : 64 * LD);   // [hd]
  float* kraw = qraw + hdp;             // [hd]
  float* wq = kraw + hdp;               // [hd]
  float* wk = wq + hdp;                 // [hd]
  float* cs = wk + hdp;                 // [hd/2]
  float* sn = cs + hdp;                 // [hd/2]
  float* sq = sn + hdp;                 // [2][hd]
  __shared__ float inv_s[2];
  int bx, h;
  attn_xcd_map(a.xcd_map, &bx, &h);
  const int t = blockIdx.z, lane = threadIdx.x;
  const int P = a.pos0 + t;
  const int tk0 = bx * 64;
  if (tk0 > P) return;
  const int group = a.nq / a.nkv;
  const int kvh = h / group;
  const float* qrow = a.qkv + (size_t)t * a.ld + (size_t)h * hd;
  const float* kbase = a.kc + ((size_t)kvh * a.max_seq + tk0) * hd;
  const int rows = min(64, P + 1 - tk0);
  const bool own_new = a.fuse_heads && P - tk0 < 64;   // this block holds row P
  const int cached = own_new ? rows - 1 : rows;        // rows read from the cache
  const int h4 = hd / 4;
  const int total = cached * h4;
  // fuse_heads: the head rows, norm weights and cos/sin into registers first
  // (a wave's loads complete in order: heads_prep below then waits for these
  // alone, not for the K rows requested after them)
  constexpr int SR = (REG ? kRegHd : kMaxHd) / 64, SC = SR / 2;
  float rq[SR], rwq[SR], rk[SR], rwk[SR], rv[SR], rcs[SC], rsn[SC];
  const bool write_v = own_new && h % group == 0;
  if (a.fuse_heads) {
    const float* krow = a.qkv + (size_t)t * a.ld + (size_t)(a.nq + kvh) * hd;
    const float* vraw = a.qkv + (size_t)t * a.ld + (size_t)(a.nq + a.nkv + kvh) * hd;
#pragma unroll
    for (int u = 0; u < SR; ++u) {
      const int d = lane + 64 * u;
      const bool in = d < hd;
      rq[u] = in ? qrow[d] : 0.0f;
      rwq[u] = in && a.q_norm ? a.q_norm[d] : 0.0f;
      rk[u] = in && own_new ? krow[d] : 0.0f;
      rwk[u] = in && own_new && a.k_norm ? a.k_norm[d] : 0.0f;
      rv[u] = in && write_v ? vraw[d] : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < SC; ++u) {
      const int i = lane + 64 * u;
      rcs[u] = i < d2 ? a.rope_cos[(size_t)P * d2 + i] : 0.0f;
      rsn[u] = i < d2 ? a.rope_sin[(size_t)P * d2 + i] : 0.0f;
    }
  }
  float4 kr[REG ? kRegHd / 4 : 1];
  if constexpr (REG) {
    // this lane's K row (position tk0 + lane) into registers
    // (columns past hd: the row's last float4 again; their products are not summed)
    const float4* src = reinterpret_cast<const float4*>(kbase + (size_t)(lane < cached ? lane : 0) * hd);
#pragma unroll
    for (int i = 0; i < kRegHd / 4; ++i) kr[i] = src[i < h4 ? i : h4 - 1];
  } else {
    // 16 loads in flight per lane, then their stores
    for (int base = 0; base < total; base += 64 * 16) {
      float4 r[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int i = base + lane + 64 * u;
        r[u] = i < total ? *reinterpret_cast<const float4*>(kbase + (size_t)(i / h4) * hd + 4 * (i % h4))
                         : zero4();
      }
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int i = base + lane + 64 * u;
        if (i < total) *reinterpret_cast<float4*>(kt + (i / h4) * LD + 4 * (i % h4)) = r[u];
      }
    }
  }
  if (a.fuse_heads) {
#pragma unroll
    for (int u = 0; u < SR; ++u) {
      const int d = lane + 64 * u;
      if (d < hd) {
        qraw[d] = rq[u];
        wq[d] = rwq[u];
        kraw[d] = rk[u];
        wk[d] = rwk[u];
      }
    }
#pragma unroll
    for (int u = 0; u < SC; ++u) {
      const int i = lane + 64 * u;
      if (i < d2) {
        cs[i] = rcs[u];
        sn[i] = rsn[u];
      }
    }
    if (write_v) {   // V row P into the cache unchanged
      float* vd = a.vc + ((size_t)kvh * a.max_seq + P) * hd;
#pragma unroll
      for (int u = 0; u < SR; ++u)
        if (lane + 64 * u < hd) vd[lane + 64 * u] = rv[u];
    }
    __syncthreads();
    float* knew = REG ? kt : kt + (P - tk0) * LD;
    heads_prep(qraw, own_new ? kraw : nullptr, a.q_norm ? wq : nullptr, a.k_norm ? wk : nullptr,
               a.eps, hd, cs, sn, sq, inv_s, q, knew);
    if (own_new && h % group == 0) {
      __syncthreads();
      float* kd = a.kc + ((size_t)kvh * a.max_seq + P) * hd;
      for (int d = lane; d < hd; d += 64) kd[d] = knew[d];
    }
  } else {
    for (int d = lane; d < hd; d += 64) q[d] = qrow[d];
  }
  __syncthreads();
  if (lane < rows) {
    float dot;
    if constexpr (REG) {
      if (own_new && lane == P - tk0) {   // row P: computed above, in LDS
        const float4* kn4 = reinterpret_cast<const float4*>(kt);
#pragma unroll
        for (int i = 0; i < kRegHd / 4; ++i) kr[i] = kn4[i < h4 ? i : h4 - 1];
      }
      const float4* q4 = reinterpret_cast<const float4*>(q);
      dot = 0.0f;
      // the query (an LDS broadcast) is read 8 float4 ahead of its adds
#pragma unroll
      for (int ib = 0; ib < kRegHd / 4; ib += 8) {
        float4 qv[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) qv[u] = q4[ib + u < h4 ? ib + u : h4 - 1];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          if (ib + u < h4) {
            const float p0 = qv[u].x * kr[ib + u].x, p1 = qv[u].y * kr[ib + u].y;
            const float p2 = qv[u].z * kr[ib + u].z, p3 = qv[u].w * kr[ib + u].w;
            dot = dot + p0;
            dot = dot + p1;
            dot = dot + p2;
            dot = dot + p3;
          }
        }
      }
    } else {
      dot = chain_dot(0.0f, q, kt + lane * LD, h4);
    }
    a.S[((size_t)t * a.nq + h) * a.max_seq + tk0 + lane] = dot * a.scale;
  }
}

constexpr int kPvThreads = 256, kPvDpb = 16;

// Softmax of the n = pos0 + t + 1 scores of (t, h) and the weighted V sum
// for head dimensions DPB*g .. DPB*g + DPB - 1 (test_model_trace.c:408-426), up
// to four query rows:
//   m = S[0], then every larger score (a NaN S[0] stays; later NaNs never
//   win); e_i = expf(S_i - m); sum = (((0 + e_0) + e_1) + ...) (the
//   sequential sum: one chain, or block_seq_sum for long rows);
//   p_i = e_i * (1 / (sum + 1e-9)); out_d = (((0 + p_0 v_0d) + p_1 v_1d) + ...).
// The weighted sum runs over chunks of CH positions: every thread forms
// products p_i * v_id of the chunk into a transposed LDS tile [d][i] (the
// next chunk's V loads already in flight), then lanes d < DPB sum their row
// with pure dependent adds.  Products past n are 0 * 0 = +0 (no-ops).
__global__ __launch_bounds__(kPvThreads) void attn_softmax_pv_kernel(AttnArgs a) {
  constexpr int DPB = kPvDpb;
  constexpr int CH = 16384 / DPB;                  // positions per chunk
  constexpr int Q4 = DPB / 4;                      // float4 per position
  constexpr int NL = CH * Q4 / kPvThreads;         // float4 per thread per chunk
  constexpr int LDT = CH + 4;
  extern __shared__ float lds[];
  const int hd = a.hd;
  int bx, h;
  attn_xcd_map(a.xcd_map, &bx, &h);
  const int t = blockIdx.z;
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const int n = a.pos0 + t + 1;
  float* es = lds;                                  // [max_seq, rounded up to 4]
  float* pt = lds + ((a.max_seq + 3) & ~3);         // [DPB][LDT]
  __shared__ float red[kPvThreads / kWave];
  __shared__ SeqSumScratch seq;
  const int kvh = h / (a.nq / a.nkv);
  const int d0 = DPB * bx;
  const int dl = min(DPB, hd - d0);
  const float* vbase = a.vc + (size_t)kvh * a.max_seq * hd + d0;
  const int nch = (n + CH - 1) / CH;
  float4 rg[NL];
  auto load = [&](int c) {
#pragma unroll
    for (int u = 0; u < NL; ++u) {
      const int i = tid + kPvThreads * u;
      const int pos = c * CH + i / Q4, q4 = i % Q4;
      rg[u] = (pos < n && 4 * q4 < dl) ? *reinterpret_cast<const float4*>(vbase + (size_t)pos * hd + 4 * q4)
                                       : zero4();
    }
  };
  auto store = [&](int c) {
#pragma unroll
    for (int u = 0; u < NL; ++u) {
      const int i = tid + kPvThreads * u;
      const int lp = i / Q4, q4 = i % Q4, pos = c * CH + lp;
      const float pk = pos < n ? es[pos] : 0.0f;
      float* col = pt + 4 * q4 * LDT + lp;
      col[0] = pk * rg[u].x;
      col[LDT] = pk * rg[u].y;
      col[2 * LDT] = pk * rg[u].z;
      col[3 * LDT] = pk * rg[u].w;
    }
  };
  // the scores first (into registers when they fit), then the first V
  // tile, which loads while the softmax runs (a thread's loads complete in
  // order, so the max waits for the scores alone)
  const float* Srow = a.S + ((size_t)t * a.nq + h) * a.max_seq;
  constexpr int SR = 8;
  const bool s_regs = n <= SR * kPvThreads;
  float sr[SR];
  if (s_regs) {
#pragma unroll
    for (int u = 0; u < SR; ++u) {
      const int i = tid + kPvThreads * u;
      sr[u] = i < n ? Srow[i] : 0.0f;
    }
  }
  load(0);
  float mx = -__builtin_inff();
  if (s_regs) {
#pragma unroll
    for (int u = 0; u < SR; ++u) {
      const int i = tid + kPvThreads * u;
      if (i < n) {
        const float s = sr[u];
        es[i] = s;
        if (s == s && s > mx) mx = s;
      }
    }
  } else {
    for (int i = tid; i < n; i += kPvThreads) {
      const float s = Srow[i];
      es[i] = s;
      if (s == s && s > mx) mx = s;
    }
  }
  // order-free max over the non-NaN scores (-inf when there is none)
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float o = __shfl_xor(mx, off, kWave);
    mx = o > mx ? o : mx;
  }
  if (lane == 0) red[wave] = mx;
  __syncthreads();
  float m = red[0];
  for (int w = 1; w < kPvThreads / kWave; ++w) m = red[w] > m ? red[w] : m;
  const float s0 = es[0];
  if (s0 != s0) m = s0;
  for (int i = tid; i < n; i += kPvThreads) es[i] = expf_glibc(es[i] - m);
  for (int i = n + tid; i < ((n + 3) & ~3); i += kPvThreads) es[i] = 0.0f;
  __syncthreads();
  // the sum: by the whole block for long rows (prefill), else one chain in
  // thread 0 (block_seq_sum's fixed cost exceeds a chain of a few hundred)
  float esum;
  if constexpr (DPB >= 128) {
    esum = block_seq_sum<kPvThreads>(es, n, seq);
  } else {
    if (tid == 0) seq.result = chain_sum(0.0f, es, (n + 3) / 4);
    __syncthreads();
    esum = seq.result;
  }
  const float inv = 1.0f / (esum + 1e-9f);
  for (int i = tid; i < n; i += kPvThreads) es[i] = es[i] * inv;
  __syncthreads();
  float out = 0.0f;
  // the next product's first chunks toward the memory-side cache (values
  // unused), requested once the V tile is in LDS so that no wait for V or
  // the scores counts them
  constexpr int PFN = kAttnPfRows * kAttnPfCols / 4 / kPvThreads;
  float4 pfv[PFN];
  const bool pf = a.pf_w && t == 0 && DPB == 16;
  for (int c = 0; c < nch; ++c) {
    store(c);
    if (c + 1 < nch) load(c + 1);
    if (c == 0 && pf) {
      const int b = (int)blockIdx.x + (int)gridDim.x * (int)blockIdx.y;
#pragma unroll
      for (int u = 0; u < PFN; ++u) {
        const int i = tid + kPvThreads * u;
        const int row = kAttnPfRows * b + i / (kAttnPfCols / 4), c4 = i % (kAttnPfCols / 4);
        pfv[u] = row < a.pf_n && 4 * c4 + 4 <= a.pf_ld
                     ? *reinterpret_cast<const float4*>(a.pf_w + (size_t)row * a.pf_ld + 4 * c4)
                     : zero4();
      }
    }
    __syncthreads();
    const int np = min(CH, n - c * CH);
    if (tid < dl) out = chain_sum(out, pt + tid * LDT, (np + 3) / 4);
    __syncthreads();
  }
  if (tid < dl) a.H[(size_t)t * a.nq * hd + (size_t)h * hd + d0 + tid] = out;
  if (pf) {
#pragma unroll
    for (int u = 0; u < PFN; ++u) asm volatile("" ::"v"(pfv[u].x));   // keeps the requests
  }
}

// ---- many query rows (prefill) ----
//
// The one-row kernels above read the whole key / value prefix once per query
// row; these read it once per 32 (scores) or 16 rows (V sums), with the
// products on the matrix cores and the chains' adds on the VALU as in
// dense_mfma_kernel (its operand layout: lane (b, j) = (lane / 16, lane % 16), MFMA c of 16 columns has
// column 4b + c in block b, result register 4b' + r of MFMA c the product of
// chain r and column 4b' + c).  Same chains, same order: bit-identical
// results.  512 rows from position 0, 32 / 4 heads of 128: scores 71 -> 32 us, V
// sums 74 -> 25 (15 of each are the products and adds at 4.3 clocks per 64),
// softmax 16.

// The head of block x of a grid whose x runs over the nq heads: blocks are
// dealt to the 8 XCDs in turn, so XCD k takes heads k nq/8 .. and a KV head's
// rows come from few XCDs' L2s.  Heads run fastest in these grids: with the key
// chunks fastest, XCD 0 took the keys that every row sees (43 us of scores
// against 34).
__device__ __forceinline__ int attn_head(int x, int nq) {
  return nq % 8 ? x : x % 8 * (nq / 8) + x / 8;
}

// Scores of query rows t0 .. t0 + 31 of one head against `tiles` tiles of 32
// keys from 32 tiles blockIdx.y on; wave w: rows 16 (w % 2) .., keys 16 (w / 2)
// .. of each tile.  The queries stay in LDS, the key
// tiles stream through a ring of D buffers in stages of 64 columns (nh stages
// a tile, columns past hd zero), so that only a block's first loads are waited
// for (512 rows, one tile a block: 45 us, most of it blocks waiting for their
// own two loads; with fewer blocks than the chip
// holds the wait for more tiles is longer than that one: 8 rows at position 250
// 11.3 -> 6.2 us, 512 rows of 4 heads 17.1 -> 16.0).  q must already be normed and rotated (heads_kernel).
// S rows (head, token) are a.ss apart; key <= pos0 + t only is written.
constexpr int kSq = 32, kSk = 32, kSktMax = 4;
constexpr int kSkD = 3;
constexpr int kStageB = 32 * 64 * 4;   // bytes of 32 rows x 64 columns

__global__ __launch_bounds__(256, 4) void attn_scores_qt_kernel(AttnArgs a, int tiles) {
  constexpr int SL = 16, NL = 2;   // 16-byte slots of a row; load instructions of a stage per wave
  extern __shared__ float4 sq4[];  // [nh] query stages, [kSkD] key stages
  const int hd = a.hd, nh = (hd + 63) / 64;
  const int h = attn_head(blockIdx.x, a.nq), tk0 = blockIdx.y * (kSk * tiles);
  const int t0 = ((int)gridDim.z - 1 - (int)blockIdx.z) * kSq;
  const int Pmax = min(a.pos0 + t0 + kSq, a.pos0 + a.T) - 1;
  if (tk0 > Pmax) return;   // every key of the block is masked (uniform)
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int b = lane / 16, j = lane % 16, wx = wave % 2, wn = wave / 2;
  const int kvh = h / (a.nq / a.nkv);
  const float* kbase = a.kc + (size_t)kvh * a.max_seq * hd;
  const int steps = min(tiles, (Pmax - tk0) / kSk + 1) * nh;
  uint8_t* qlds = reinterpret_cast<uint8_t*>(sq4);
  uint8_t* klds = qlds + nh * kStageB;
  // instruction v of a stage: rows 4 (wave + 4v) + lane / 16
  int row[NL], col[NL];
#pragma unroll
  for (int v = 0; v < NL; ++v) {
    row[v] = 4 * (wave + 4 * v) + lane / SL;
    col[v] = 4 * ((lane % SL) ^ (row[v] & 15));
  }
  auto load_k = [&](int s, int buf) {
    const int key0 = tk0 + kSk * (s / nh), c0 = 64 * (s % nh);
#pragma unroll
    for (int v = 0; v < NL; ++v)
      lds_load16(c0 + col[v] < hd ? kbase + (size_t)min(key0 + row[v], Pmax) * hd + c0 + col[v] : kDenseZero,
                 klds + buf * kStageB + (wave + 4 * v) * 1024);
  };
  for (int c = 0; c < nh; ++c)
#pragma unroll
    for (int v = 0; v < NL; ++v)
      lds_load16(64 * c + col[v] < hd
                     ? a.qkv + (size_t)min(t0 + row[v], a.T - 1) * a.ld + (size_t)h * hd + 64 * c + col[v]
                     : kDenseZero,
                 qlds + c * kStageB + (wave + 4 * v) * 1024);
#pragma unroll
  for (int p = 0; p < kSkD - 1; ++p) load_k(min(p, steps - 1), p);
  float acc[4] = {}, done[4];
  auto put = [&](int tile) {   // the finished tile's scores
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int tok = t0 + 16 * wx + 4 * b + r, key = tk0 + kSk * tile + 16 * wn + j;
      if (tok < a.T && key <= a.pos0 + tok) a.S[((size_t)h * a.T + tok) * a.ss + key] = done[r] * a.scale;
    }
  };
  for (int s = 0; s < steps; ++s) {
    stage_sync<(kSkD - 2) * NL>();
    // a tile's stores go out before the next loads, so that the wait above
    // counts them only a whole stage later
    if (s && s % nh == 0) put(s / nh - 1);
    load_k(min(s + kSkD - 1, steps - 1), (s + kSkD - 1) % kSkD);
    const float4* Q = reinterpret_cast<const float4*>(qlds + (s % nh) * kStageB) + (16 * wx + j) * SL;
    const float4* B = reinterpret_cast<const float4*>(klds + (s % kSkD) * kStageB) + (16 * wn + j) * SL;
    float4 x = Q[b ^ j], w = B[b ^ j];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      float4 xn = x, wn4 = w;
      if (g + 1 < 4) {
        xn = Q[(4 * (g + 1) + b) ^ j];
        wn4 = B[(4 * (g + 1) + b) ^ j];
      }
      asm volatile("" ::: "memory");
      v16f p[4];
      mfma_products(x, w, p);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < 16; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = acc[r] + p[k % 4][4 * (k / 4) + r];
      __builtin_amdgcn_sched_barrier(0);
      x = xn;
      w = wn4;
    }
    if (s % nh == nh - 1) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        done[r] = acc[r];
        acc[r] = 0.0f;
      }
    }
  }
  put((steps - 1) / nh);
  stage_sync<0>();   // the clamped loads past the last stage have landed
}

// Softmax of the score rows, in place (test_model_trace.c:411-420): a block
// takes R query rows of a head, n = pos0 + t + 1 scores each, staged in LDS
// (the longest rows' blocks first, those of one length spread over the CUs);
// max per row by one wave (order-free; a NaN first score wins, as in
// attn_softmax_pv_kernel), e = expf(s - m), then lane i of wave 0 runs row
// i's sum chain, and p = e * (1 / (sum + 1e-9)) goes back over the scores.  A
// row a wave: 16 rows a block left each wave four rows to exponentiate one
// after another (32 heads: 16 rows at position 250 9.6 -> 5.2 us, 8 at 1000 14.5
// -> 10.2, 512 at 0 .. 1500 49 -> 36; two rows 51, one row 80).
constexpr int kSmRowsMax = 4;

// Floats of a staged row: whole 256-float load instructions, and four so that
// the 16 lanes of a chain read meet different banks.
__host__ __device__ constexpr int sm_row_floats(int npos) { return (npos + 255) / 256 * 256 + 4; }

__global__ __launch_bounds__(256) void attn_softmax_rows_kernel(AttnArgs a, int R) {
  extern __shared__ float smr[];   // [R][LD]
  __shared__ float inv_s[kSmRowsMax];
  __shared__ uint64_t exp_tab[32];
  if (threadIdx.x < 32) exp_tab[threadIdx.x] = kExp2Tab[threadIdx.x];
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int LD = sm_row_floats(a.pos0 + a.T);
  const int h = attn_head(blockIdx.x, a.nq), t0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * R;
  const int nr = min(R, a.T - t0);
  float* S0 = a.S + ((size_t)h * a.T + t0) * a.ss;
  for (int i = wave; i < nr; i += 4) {
    const int n = a.pos0 + t0 + i + 1;
    const float* Srow = S0 + (size_t)i * a.ss;
    for (int c = 0; c < n; c += 256)
      lds_load16(c + 4 * lane < a.ss ? Srow + c + 4 * lane : kDenseZero,
                 reinterpret_cast<uint8_t*>(smr + (size_t)i * LD + c));
  }
  stage_sync<0>();
  for (int i = wave; i < nr; i += 4) {
    const int n = a.pos0 + t0 + i + 1;
    float* er = smr + (size_t)i * LD;
    const float s0 = er[0];
    float mx = -__builtin_inff();
    for (int k = lane; k < n; k += kWave) {
      const float v = er[k];
      if (v == v && v > mx) mx = v;
    }
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
      const float o = __shfl_xor(mx, off, kWave);
      mx = o > mx ? o : mx;
    }
    const float m = s0 != s0 ? s0 : mx;
    // four exponentials side by side (LDS reads, table lookups and fp64 chains)
    int k = lane;
    for (; k + 3 * kWave < n; k += 4 * kWave) {
      float e[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) e[u] = er[k + u * kWave] - m;
#pragma unroll
      for (int u = 0; u < 4; ++u) e[u] = expf_glibc_t(e[u], exp_tab);
#pragma unroll
      for (int u = 0; u < 4; ++u) er[k + u * kWave] = e[u];
    }
    for (; k < n; k += kWave) er[k] = expf_glibc_t(er[k] - m, exp_tab);
    if (lane < 3 && n + lane < ((n + 3) & ~3)) er[n + lane] = 0.0f;
  }
  __syncthreads();
  if ((int)threadIdx.x < nr) {
    const int n = a.pos0 + t0 + (int)threadIdx.x + 1;
    inv_s[threadIdx.x] = 1.0f / (chain_sum(0.0f, smr + (size_t)threadIdx.x * LD, (n + 3) / 4) + 1e-9f);
  }
  __syncthreads();
  for (int i = wave; i < nr; i += 4) {
    const int n = a.pos0 + t0 + i + 1;
    float* Srow = S0 + (size_t)i * a.ss;
    const float* er = smr + (size_t)i * LD;
    const float inv = inv_s[i];
    for (int k = lane; k < n; k += kWave) Srow[k] = er[k] * inv;
  }
}

// Weighted V sums of query rows t0 .. t0 + 15 of one head for dimensions 64
// blockIdx.y ..; wave w: dimensions 16 w .. of those.  out = (((0 + p_0 v_0) + p_1 v_1) + ...) over a row's n = pos0 + t + 1
// positions: chunks of kPvCh positions of p (rows a.ss apart) and V stream
// through two LDS buffers; a product past the row's n counts as +0, which
// leaves its chain unchanged (a chain from +0 is never -0).  The longest
// rows' blocks come first in the grid.  One 16 x 16 tile of products a step and
// wave: two (32 rows a block) double the chain of a launch that a few rows
// leave waiting, and cost the full chip a block a CU in registers (32 / 4 heads
// of 128, 8 rows at position 1000: 32.2 -> 20.9 us, 64 rows 36.7 -> 24.4, 512
// rows at 1000 .. 72.6 -> 68.7).
constexpr int kPvCh = 32, kPvR = 16;

__global__ __launch_bounds__(256, 4) void attn_pv_qt_kernel(AttnArgs a) {
  constexpr int PS = kPvCh / 4, VS = 16;                  // 16-byte slots of a p row, a V row (64 dimensions)
  constexpr int NP = kPvR * PS / 64, NV = kPvCh * VS / 64; // load instructions
  static_assert(NP == 2 && NV == 8, "one of the first two waves, two of every wave");
  __shared__ float4 lds4[2][kPvR * PS + kPvCh * VS];
  const int hd = a.hd, h = attn_head(blockIdx.x, a.nq), d0 = blockIdx.y * 64;
  const int t0 = ((int)gridDim.z - 1 - (int)blockIdx.z) * kPvR;
  const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
  const int b = lane / 16, j = lane % 16;
  const int nmax = min(a.pos0 + t0 + kPvR, a.pos0 + a.T);  // positions of the last row
  const int nc = (nmax + kPvCh - 1) / kPvCh;
  const int kvh = h / (a.nq / a.nkv);
  // instruction `wave` < NP loads p rows (8 each), NP + wave and NP + 4 + wave V
  // rows (4 each)
  const int prow = 8 * wave + lane / PS, pcol = 4 * ((lane % PS) ^ ((prow >> 1) & 7));
  const float* psrc = a.S + ((size_t)h * a.T + min(t0 + prow, a.T - 1)) * a.ss + pcol;
  const float* vbase = a.vc + (size_t)kvh * a.max_seq * hd;
  // V slot s of row r sits at s ^ 4 (r >> 2 & 3): the four blocks' rows 4b + c
  // then meet four different quarters of the banks
  int vrow[2], vcol[2];
#pragma unroll
  for (int v = 0; v < 2; ++v) {
    vrow[v] = 4 * (wave + 4 * v) + lane / VS;
    vcol[v] = d0 + 4 * ((lane % VS) ^ (4 * ((vrow[v] >> 2) & 3)));
  }
  auto load = [&](int c, int half) {
    uint8_t* l = reinterpret_cast<uint8_t*>(lds4[half]);
    const int c0 = c * kPvCh;
    if (wave < NP) lds_load16(c0 + pcol < a.ss ? psrc + c0 : kDenseZero, l + wave * 1024);
#pragma unroll
    for (int v = 0; v < 2; ++v)
      lds_load16(vcol[v] < hd ? vbase + (size_t)min(c0 + vrow[v], nmax - 1) * hd + vcol[v] : kDenseZero,
                 l + (NP + wave + 4 * v) * 1024);
  };
  const int nlo = a.pos0 + t0 + 1, nhi = nlo + 15;   // positions of the first and the last row
  float acc[4] = {};
  load(0, 0);
  for (int c = 0; c < nc; ++c) {
    stage_sync<0>();
    if (c + 1 < nc) load(c + 1, (c + 1) & 1);
    const float4* P = lds4[c & 1] + j * PS;
    const float* V = reinterpret_cast<const float*>(lds4[c & 1] + kPvR * PS);
#pragma unroll
    for (int g = 0; g < kPvCh / 16; ++g) {
      const int pos = c * kPvCh + 16 * g;
      if (pos >= nhi) break;
      const float4 x = P[(4 * g + b) ^ ((j >> 1) & 7)];
      const float* v = V + (16 * g + 4 * b) * 64 + 4 * ((4 * wave + j / 4) ^ (4 * b)) + j % 4;
      const float4 w = make_float4(v[0], v[64], v[128], v[192]);
      v16f p[4];
      mfma_products(x, w, p);
      if (pos + 16 > nlo) {
        const int left = nlo + 4 * b - pos;   // row r: left + r positions from pos on
#pragma unroll
        for (int k = 0; k < 16; ++k)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float q = p[k % 4][4 * (k / 4) + r];
            p[k % 4][4 * (k / 4) + r] = k < left + r ? q : 0.0f;
          }
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < 16; ++k)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[r] = acc[r] + p[k % 4][4 * (k / 4) + r];
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int tok = t0 + 4 * b + r, d = d0 + 16 * wave + j;
    if (tok < a.T && d < hd) a.H[(size_t)tok * a.nq * hd + (size_t)h * hd + d] = acc[r];
  }
}

// ---------------------------------------------------------------- misc

__global__ __launch_bounds__(256) void embed_kernel(const int32_t* __restrict__ ids,
                                                    const float* __restrict__ emb, int V, int D,
                                                    float* __restrict__ x) {
  const int t = blockIdx.x;
  int id = ids[t];
  id = id < 0 ? 0 : (id >= V ? V - 1 : id);
  const float* src = emb + (size_t)id * D;
  float* dst = x + (size_t)t * D;
  for (int i = threadIdx.x; i < D; i += 256) dst[i] = src[i];
}

constexpr int kGreedyThreads = 1024;

// The smallest v over the block (all threads get it); red: one int per wave.
__device__ int block_min(int v, int* red) {
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const int o = __shfl_xor(v, off, kWave);
    v = o < v ? o : v;
  }
  __syncthreads();
  if (lane == 0) red[wave] = v;
  __syncthreads();
  for (int w = 0; w < (int)blockDim.x / kWave; ++w) v = red[w] < v ? red[w] : v;
  return v;
}

// The reference's next token (test_model_trace.c:735-746): softmax_rows of
// the logits, then the first index of the largest probability.  With m the
// largest logit: a NaN or +inf logit, or m = -inf, turns every probability
// into NaN and the scan stays at 0.  Otherwise e_i = expf(v_i - m) <= 1
// with e = 1 at the maximum, the probabilities are e_i * inv with a normal
// inv = 1 / (sum + 1e-9) (sum >= 1), and any e_i <= 1 - 2^-24 gives a
// product that rounds below inv (the exact (1 - 2^-24) inv is at least
// half an ulp of inv under it, and exactly representable when it is only
// that), so the answer is the first i with expf(v_i - m) == 1.
// part (optional): the largest value of every block of `rows` consecutive
// logits (NaN if the block holds one), written by the head's product; only
// the first block whose maximum qualifies is then scanned.
__global__ __launch_bounds__(kGreedyThreads) void greedy_kernel(const float* __restrict__ v, int n,
                                                               const float* __restrict__ part,
                                                               int rows, int32_t* out,
                                                               int32_t* hist, int32_t* hist_pos) {
  __shared__ float fred[kGreedyThreads / kWave];
  __shared__ int ired[kGreedyThreads / kWave];
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  const float* src = part ? part : v;
  const int ns = part ? (n + rows - 1) / rows : n;
  // up to GR values a thread are loaded at once and kept in registers for
  // both scans (a loop of dependent loads costs a round trip per value)
  constexpr int GR = 12;
  const bool in_regs = ns <= GR * kGreedyThreads;
  float sv[GR];
  float mx = -__builtin_inff();
  if (in_regs) {
#pragma unroll
    for (int u = 0; u < GR; ++u) {
      const int i = tid + kGreedyThreads * u;
      sv[u] = i < ns ? src[i] : -__builtin_inff();
    }
#pragma unroll
    for (int u = 0; u < GR; ++u) mx = nan_max(mx, sv[u]);
  } else {
    for (int i = tid; i < ns; i += kGreedyThreads) mx = nan_max(mx, src[i]);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mx = nan_max(mx, __shfl_xor(mx, off, kWave));
  if (lane == 0) fred[wave] = mx;
  __syncthreads();
  float m = fred[0];
  for (int w = 1; w < kGreedyThreads / kWave; ++w) m = nan_max(m, fred[w]);
  int ans = 0;
  if (m == m && m != __builtin_inff() && m != -__builtin_inff()) {
    int first = INT_MAX;
    if (in_regs) {
#pragma unroll
      for (int u = GR - 1; u >= 0; --u) {
        // (d < -1e-6: e^d < 1 - 9.9e-7, 16 ulps under 1, so expf(d) < 1)
        const int i = tid + kGreedyThreads * u;
        const float d = sv[u] - m;
        if (i < ns && !(d < -1e-6f) && expf_glibc(d) == 1.0f) first = i;
      }
    } else {
      for (int i = tid; i < ns; i += kGreedyThreads)
        if (expf_glibc(src[i] - m) == 1.0f) { first = i; break; }
    }
    first = block_min(first, ired);
    if (part && first != INT_MAX) {
      const int lo = first * rows, hi = min(n, lo + rows);
      first = INT_MAX;
      for (int i = lo + tid; i < hi; i += kGreedyThreads)
        if (expf_glibc(v[i] - m) == 1.0f) { first = i; break; }
      first = block_min(first, ired);
    }
    ans = first == INT_MAX ? 0 : first;
  }
  if (tid == 0) {
    out[0] = ans;
    if (hist) {
      const int p = *hist_pos;
      hist[p] = ans;
      *hist_pos = p + 1;
    }
  }
}

constexpr int kSmThreads = 1024;
constexpr int kSmChunk = 8192;

// softmax_rows (test_model_trace.c:260-272) of one row in place: max as in
// the attention softmax, e_i = expf(v_i - max) in parallel, the sum as one
// chain over LDS-staged chunks, then v_i = e_i * (1 / (sum + 1e-9)).
__global__ __launch_bounds__(kSmThreads) void softmax_vec_kernel(float* v, int n) {
  __shared__ float chunk[kSmChunk];
  __shared__ float red[kSmThreads / kWave];
  __shared__ float inv_s;
  const int tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
  float mx = -__builtin_inff();
  for (int i = tid; i < n; i += kSmThreads) {
    const float s = v[i];
    if (s == s && s > mx) mx = s;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const float o = __shfl_xor(mx, off, kWave);
    mx = o > mx ? o : mx;
  }
  if (lane == 0) red[wave] = mx;
  __syncthreads();
  float m = red[0];
  for (int w = 1; w < kSmThreads / kWave; ++w) m = red[w] > m ? red[w] : m;
  const float v0 = v[0];
  if (v0 != v0) m = v0;
  __syncthreads();
  float sum = 0.0f;
  for (int base = 0; base < n; base += kSmChunk) {
    const int len = min(kSmChunk, n - base);
    for (int i = tid; i < len; i += kSmThreads) {
      const float e = expf_glibc(v[base + i] - m);
      chunk[i] = e;
      v[base + i] = e;
    }
    __syncthreads();
    if (tid == 0)
      for (int i = 0; i < len; ++i) sum = sum + chunk[i];
    __syncthreads();
  }
  if (tid == 0) inv_s = 1.0f / (sum + 1e-9f);
  __syncthreads();
  const float inv = inv_s;
  for (int i = tid; i < n; i += kSmThreads) v[i] = v[i] * inv;
}

bool al16(const void* p) { return ((uintptr_t)p & 15) == 0; }

// Dynamic LDS above 64 KB needs the kernel's attribute raised; the largest
// size set per kernel is remembered so the runtime is called once per size.
std::mutex g_lds_mu;
std::unordered_map<const void*, size_t> g_lds_set;

template <class F>
moe_status set_lds(F* fn, size_t bytes, const char* what) {
  if (bytes <= 65536) return MOE_OK;
  std::lock_guard<std::mutex> lk(g_lds_mu);
  size_t& cur = g_lds_set[(const void*)fn];
  if (bytes <= cur) return MOE_OK;
  moe_status st = check_hip(hipFuncSetAttribute((const void*)fn,
                                                hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes),
                            what);
  if (st == MOE_OK) cur = bytes;
  return st;
}

template <int WX, int NB, int KC, int D, bool ANY>
moe_status launch_mfma(const DenseArgs& a, hipStream_t s) {
  constexpr int RX = 16 * WX, RW = 16 * NB * (4 / WX);
  dim3 grid((unsigned)((a.N + RW - 1) / RW), (unsigned)((a.M + RX - 1) / RX));
  hipLaunchKernelGGL((dense_mfma_kernel<WX, NB, KC, D, ANY>), grid, dim3(256), 0, s, a);
  return check_hip(hipGetLastError(), "dense mfma launch");
}

// The tile shape with the least estimated time.  Per column of K a CU with m
// blocks takes about step * m clocks, and `odd` more when m is odd (a SIMD's
// last wave runs alone: 6.6 clocks per 64 products against 4.5 for two).
// Measured, clocks per column at K = 2048 and 4096: 32 x 32 tiles 37, 55, 73,
// 88, 234 for m = 1, 2, 3, 4, 10; 32 x 64 65, 91, 131, 210 for m = 1, 2, 3, 5;
// 64 x 64 116, 160, 246, 586 for m = 1, 2, 3, 8; 64 x 80 145, 199, 305 for m =
// 1, 2, 3.  Small tiles spread few tokens over the CUs, large ones spend less
// on operands per product.
// A grid holds 65535 row tiles: taller products keep the 64-row shapes (up to
// 4,194,240 rows); -1 past those.
// *t: the estimate, clocks per column.
int mfma_shape(int M, int N, double* t_out) {
  struct Shape { int rx, rw, step, odd; };
  static const Shape shapes[4] = {{32, 32, 22, 10}, {32, 64, 40, 18}, {64, 64, 75, 42}, {64, 80, 95, 50}};
  int best = -1;
  double tbest = 0.0;
  for (int i = 0; i < 4; ++i) {
    const Shape& h = shapes[i];
    const long long tiles = ((long long)M + h.rx - 1) / h.rx;
    if (tiles > 65535) continue;
    const long long m = (((long long)N + h.rw - 1) / h.rw * tiles + 255) / 256;
    const double t = (double)m * h.step + (m & 1) * h.odd;
    if (best < 0 || t < tbest) { best = i; tbest = t; }
  }
  *t_out = tbest;
  return best;
}

// 5-16 tokens: whether the chain kernel (launch_gemv<4>) takes less time than
// the tiles.  Its blocks of four rows run per CU as their LDS allows and take
// about 4 + M clocks a column (M chains side by side), 8% more for each
// neighbour, and 7200 around that; the tiles 6000 around theirs.  Measured /
// estimated us, chain and tiles: 9 x 2048 x 2048 14 / 15 and 30 / 30; 8 x 5120 x
// 2048 36 / 41 and 31 / 30; 12 x 64 x 8192 56 / 58 and 111 / 112; 16 x 2048 x
// 1024 22 / 23 and 16 / 16; 12 x 2048 x 64 8 / 7 and 3 / 3.
bool chain_beats_mfma(int M, int N, int K, double t_mfma) {
  const int per_cu = M <= 6 ? 3 : M <= 9 ? 2 : 1;
  const long long rounds = (((long long)N + 3) / 4 + 256 * per_cu - 1) / (256 * per_cu);
  return (double)rounds * (K * (4.0 + M) * (0.92 + 0.08 * per_cu) + 7200.0) <= K * t_mfma + 6000.0;
}

template <bool ANY>
moe_status launch_mfma_best(const DenseArgs& a, int shape, hipStream_t s) {
  switch (shape) {
    case 0: return launch_mfma<2, 1, 64, 2, ANY>(a, s);
    case 1: return launch_mfma<2, 2, 32, 2, ANY>(a, s);
    case 2: return launch_mfma<4, 4, 32, 2, ANY>(a, s);
    default: return launch_mfma<4, 5, 32, 2, ANY>(a, s);
  }
}

size_t gemv_lds(int RW, int NP, int M, int K, bool norm) {
  const int KC = RW >= 16 ? 4096 / RW : 256;
  return ((size_t)(NP + 1) * M * RW * (KC + 4) + (norm ? (size_t)M * K : 0)) * 4;
}

template <int RW, bool NORM, int PACK, int NP, int MMX = 64 / RW>
moe_status launch_gemv(const DenseArgs& a, hipStream_t s) {
  const int groups = RW == 1 ? (a.M + MMX - 1) / MMX : 1;
  const size_t lds = gemv_lds(RW, NP, groups > 1 ? MMX : a.M, a.K, NORM);
  moe_status st = set_lds(dense_gemv_kernel<RW, NORM, PACK, NP, MMX>, lds, "gemv LDS attribute");
  if (st) return st;
  hipLaunchKernelGGL((dense_gemv_kernel<RW, NORM, PACK, NP, MMX>),
                     dim3((unsigned)((a.N + RW - 1) / RW), (unsigned)groups), dim3(64 * (NP + 1)), lds, s, a);
  return check_hip(hipGetLastError(), "dense gemv launch");
}

}  // namespace

// Producer waves of the few-token GEMV: three for one token (the LDS of four
// product buffers fits), one otherwise; the wide one-token products (the
// vocabulary head) keep three as well: their rows stream from HBM and more
// producers keep more bytes in flight.
constexpr int kNpOne = 3;
constexpr int kNpWide = 3;

bool dense_norm_ok(int M, int K) {
  return M >= 1 && M <= 4 && K % 4 == 0 && K <= 8192 &&
         gemv_lds(16, M == 1 ? kNpOne : 1, M, K, true) <= 150 * 1024;
}

// The last block selects with one wave per token, keys (8 bytes per
// logit, up to 1024) in the product buffers.
bool dense_select_ok(int M, int N) { return M >= 1 && M <= 4 && N <= 1024; }

bool dense_amax_ok(const DenseArgs& a) {
  return a.M == 1 && a.K > 0 && a.K % 4 == 0 && a.lda % 4 == 0 && a.ldw % 4 == 0 && al16(a.A) &&
         al16(a.W) && !a.norm && !a.sel_counter;
}

// 16 rows a block also for the vocabulary head: each chunk then reads 1 KB
// of every row (64-row blocks read 256 B pieces), measured ~0.4% faster per
// decode token even though the greedy choice then reads 4x the block maxima.
int dense_amax_rows(int) { return 16; }

// One token against few rows: the row kernel.
// Row kernel: one token, or up to 4 without the fused rmsnorm and packing.
bool dense_row_ok(const DenseArgs& a, bool vec) {
  const bool rows = a.M == 1 || (a.M <= 4 && !a.norm);
  return rows && a.N <= 1024 && vec && a.K <= kRowMaxK && !a.amax_part;
}

// The block-parallel rows kernel instead of the chain kernel for 5-16
// given rows (MOEHIP_ROUTER_ROWS4=1, for comparison).
bool rows4_kernel_chosen() {
  static const bool v = getenv("MOEHIP_ROUTER_ROWS4") != nullptr;
  return v;
}

// Given rows against few rows (the router): 5-16 on either rows kernel, 17-32
// against up to 256 rows (one round of blocks) on the chain kernel as two
// groups of blocks, where the 32 x 32 MFMA tiles run on a few CUs and the
// packing takes a launch of its own (Q8 layer of 20 tokens 209 -> 127 us, Q4
// 162 -> 79).
bool dense_rows4_ok(const DenseArgs& a, bool vec) {
  if (a.M > 16 && (a.M > 32 || a.N > 256 || rows4_kernel_chosen())) return false;
  return a.M > 4 && !a.norm && !a.sel_counter && !a.amax_part && a.N <= 1024 && vec &&
         a.K <= kRowsMaxK;
}

bool dense_rows4_path(const DenseArgs& a) {
  const bool vec = a.K > 0 && a.K % 4 == 0 && a.lda % 4 == 0 && a.ldw % 4 == 0 && al16(a.A) &&
                   al16(a.W);
  return a.N > 0 && dense_rows4_ok(a, vec);
}

bool dense_row_path(const DenseArgs& a) {
  const bool vec = a.K > 0 && a.K % 4 == 0 && a.lda % 4 == 0 && a.ldw % 4 == 0 && al16(a.A) &&
                   al16(a.W);
  return a.N > 0 && dense_row_ok(a, vec) && (!a.norm || dense_norm_ok(a.M, a.K));
}

template <bool NORM, int PACK>
moe_status launch_row(const DenseArgs& a, hipStream_t s) {
  const size_t lds = (size_t)2 * a.K * 4;
  moe_status st = set_lds(dense_row_kernel<NORM, PACK>, lds, "row kernel LDS attribute");
  if (st) return st;
  hipLaunchKernelGGL((dense_row_kernel<NORM, PACK>), dim3((unsigned)a.N, (unsigned)a.M), dim3(kRowThreads), lds,
                     s, a);
  if ((st = check_hip(hipGetLastError(), "dense row launch"))) return st;
  if (!a.sel_counter || a.sel_defer) return MOE_OK;
  hipLaunchKernelGGL(row_finish_kernel, dim3(1), dim3(kWave * a.M), 0, s, a);
  return check_hip(hipGetLastError(), "row finish launch");
}

moe_status dense_matmul(const DenseArgs& a, hipStream_t s) {
  if (a.M <= 0 || a.N <= 0) return MOE_OK;
  if (a.amax_part) {
    if (!dense_amax_ok(a))
      return set_error(MOE_ERR_ARG, "dense matmul: block maxima need one aligned row");
    return launch_gemv<16, false, 0, kNpOne>(a, s);
  }
  if (a.sel_counter && (!dense_select_ok(a.M, a.N) || a.sel_topk < 1 || a.sel_topk > kMaxTopK ||
                        a.ldc != a.N))
    return set_error(MOE_ERR_ARG, "dense matmul: fused selection needs M <= 4, N <= 1024");
  if (a.K <= 0) return set_error(MOE_ERR_ARG, "dense matmul: K = %d", a.K);
  if (a.sel_defer && (!a.sel_counter || !dense_row_path(a)))
    return set_error(MOE_ERR_ARG, "dense matmul: a deferred selection needs the row kernel");
  const bool vec = a.K % 4 == 0 && a.lda % 4 == 0 && a.ldw % 4 == 0 && al16(a.A) && al16(a.W);
  if (a.norm) {
    if (!vec || !dense_norm_ok(a.M, a.K))
      return set_error(MOE_ERR_ARG, "dense matmul: fused rmsnorm needs M <= 4 aligned rows");
    if (a.pack_dtype && (!a.sel_counter || !a.pack_part || !a.pack_tabs))
      return set_error(MOE_ERR_ARG, "dense matmul: packing needs the fused selection");
    if (dense_row_ok(a, vec)) {
      if (a.pack_dtype == 2) return launch_row<true, 2>(a, s);
      if (a.pack_dtype == 3) return launch_row<true, 3>(a, s);
      return launch_row<true, 0>(a, s);
    }
    if (a.M == 1) {
      if (a.pack_dtype == 2) return launch_gemv<16, true, 2, kNpOne>(a, s);
      if (a.pack_dtype == 3) return launch_gemv<16, true, 3, kNpOne>(a, s);
      // 8 rows a block: twice the blocks of the 16-row shape that the
      // packing paths keep (the [Wq;Wk;Wv] product 17.5 -> 16.9-17.2 us);
      // its four buffers (8320 floats) hold the squares of a row of K <= 8320
      if (a.K <= (kNpOne + 1) * 8 * 260) return launch_gemv<8, true, 0, kNpOne, 1>(a, s);
      return launch_gemv<16, true, 0, kNpOne>(a, s);
    }
    if (a.pack_dtype == 2) return launch_gemv<16, true, 2, 1>(a, s);
    if (a.pack_dtype == 3) return launch_gemv<16, true, 3, 1>(a, s);
    return launch_gemv<16, true, 0, 1>(a, s);
  }
  double t_mfma = 0.0;
  const int mfma = mfma_shape(a.M, a.N, &t_mfma);
  // unaligned: the tiles, but a thread an output for a few short rows (thread /
  // tiles: 16 x 1000 x 7 2.9 / 4.0 us, 300 x 2048 x 5 4.4 / 6.0, 300 x 5120 x 5 7.4 /
  // 6.5, 300 x 256 x 13 3.7 / 4.1, 32 x 5120 x 13 4.9 / 4.2, 16 x 1000 x 21 3.7 / 4.0,
  // 33 x 2048 x 21 4.9 / 4.1)
  const long long thread_work = a.K < 8 ? 4 << 20 : a.K < 16 ? 3 << 19 : a.K < 24 ? 1 << 20 : 0;
  const bool few_products = (long long)a.M * a.N <= thread_work / a.K;
  if (!vec && a.K >= 4 && mfma >= 0 && !few_products) return launch_mfma_best<true>(a, mfma, s);
  if (!vec || mfma < 0) {
    const long long total = (long long)a.M * a.N;
    hipLaunchKernelGGL(dense_generic_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, s, a);
    return check_hip(hipGetLastError(), "dense generic launch");
  }
  if (a.pack_dtype && (!a.pack_part || !a.pack_tabs ||
                       !((a.sel_counter && dense_row_ok(a, vec)) || dense_rows4_ok(a, vec))))
    return set_error(MOE_ERR_ARG, "dense matmul: packing given rows needs the row kernel and the fused "
                                  "selection, or the 5-32 token rows kernel");
  if (dense_row_ok(a, vec)) {
    if (a.pack_dtype == 2) return launch_row<false, 2>(a, s);
    if (a.pack_dtype == 3) return launch_row<false, 3>(a, s);
    return launch_row<false, 0>(a, s);
  }
  if (dense_rows4_ok(a, vec) && !rows4_kernel_chosen()) {
    // 5-32 given rows against few rows (the router): one block per row (and
    // group of 16), one
    // consumer lane per token's sequential chain, three producer waves
    if (a.pack_dtype == 2) return launch_gemv<1, false, 2, 3, 16>(a, s);
    if (a.pack_dtype == 3) return launch_gemv<1, false, 3, 3, 16>(a, s);
    return launch_gemv<1, false, 0, 3, 16>(a, s);
  }
  if (dense_rows4_ok(a, vec)) {
    const size_t lds = (size_t)kRowGroups * a.K * 4;
    const dim3 grid((unsigned)a.N, (unsigned)((a.M + kRowGroups - 1) / kRowGroups));
    moe_status st;
    if (a.pack_dtype == 2) {
      if ((st = set_lds(dense_rows4_kernel<2>, lds, "rows kernel LDS attribute"))) return st;
      hipLaunchKernelGGL(dense_rows4_kernel<2>, grid, dim3(kRowThreads), lds, s, a);
    } else if (a.pack_dtype == 3) {
      if ((st = set_lds(dense_rows4_kernel<3>, lds, "rows kernel LDS attribute"))) return st;
      hipLaunchKernelGGL(dense_rows4_kernel<3>, grid, dim3(kRowThreads), lds, s, a);
    } else {
      if ((st = set_lds(dense_rows4_kernel<0>, lds, "rows kernel LDS attribute"))) return st;
      hipLaunchKernelGGL(dense_rows4_kernel<0>, grid, dim3(kRowThreads), lds, s, a);
    }
    return check_hip(hipGetLastError(), "dense rows launch");
  }
  if (a.sel_counter) {
    if (!vec) return set_error(MOE_ERR_ARG, "dense matmul: fused selection needs aligned rows");
    return a.M == 1 ? launch_gemv<16, false, 0, kNpOne>(a, s) : launch_gemv<16, false, 0, 1>(a, s);
  }
  if (a.M == 1 && a.N >= 65536) {
    return launch_gemv<64, false, 0, kNpWide>(a, s);
  } else if (a.M <= 2 && a.N >= 32768) {
    return launch_gemv<32, false, 0, 1>(a, s);
  } else if (a.M == 1) {
    // 8 rows a block (the Wo product: 128 -> 256 blocks, 18.0 -> 17.0-17.6 us)
    return launch_gemv<8, false, 0, kNpOne, 1>(a, s);
  } else if (a.M <= 4) {
    return launch_gemv<16, false, 0, 1>(a, s);
  } else if (a.M <= 16 && chain_beats_mfma(a.M, a.N, a.K, t_mfma)) {
    return launch_gemv<4, false, 0, 1>(a, s);
  } else {
    return launch_mfma_best<false>(a, mfma, s);
  }
}

moe_status embed_rows(const int32_t* ids, int T, const float* emb, int V, int D, float* x,
                      hipStream_t s) {
  if (T <= 0) return MOE_OK;
  hipLaunchKernelGGL(embed_kernel, dim3((unsigned)T), dim3(256), 0, s, ids, emb, V, D, x);
  return check_hip(hipGetLastError(), "embed launch");
}

template <int RW>
static moe_status launch_heads(const HeadArgs& a, long long rows, hipStream_t s) {
  const size_t lds = (size_t)2 * 4 * RW * (a.hd + 4) * 4;
  moe_status st = set_lds(heads_kernel<RW>, lds, "heads LDS attribute");
  if (st) return st;
  hipLaunchKernelGGL(heads_kernel<RW>, dim3((unsigned)((rows + 4 * RW - 1) / (4 * RW))), dim3(256), lds, s, a);
  return check_hip(hipGetLastError(), "heads launch");
}

moe_status heads_norm_rope(const HeadArgs& a, hipStream_t s) {
  if (a.T <= 0) return MOE_OK;
  if (a.hd > kMaxHd || (a.hd & 1)) return set_error(MOE_ERR_ARG, "head_dim %d unsupported", a.hd);
  const long long rows = (long long)a.T * (a.nq + 2 * a.nkv);
  return rows < 4096 ? launch_heads<1>(a, rows, s) : launch_heads<4>(a, rows, s);
}

moe_status attention_rows(const AttnArgs& a, hipStream_t s) {
  if (a.T <= 0) return MOE_OK;
  if (a.hd % 4 || a.hd > kMaxHd) return set_error(MOE_ERR_ARG, "attention: head_dim %d", a.hd);
  if (a.fuse_heads && a.T != 1) return set_error(MOE_ERR_ARG, "attention: fused heads need T == 1");
  if (a.T > 4) {
    if (a.nkv <= 0 || a.nq % a.nkv || a.ss % 4 || a.ld % 4 || !al16(a.qkv))
      return set_error(MOE_ERR_ARG, "attention: many rows need whole head groups and 16-byte aligned rows");
    const unsigned qg = (unsigned)((a.T + kSq - 1) / kSq);
    const int keys = a.pos0 + a.T;
    // fewer key tiles a block where four would leave under 1024 blocks
    int tiles = kSktMax;
    while (tiles > 1 && (long long)a.nq * qg * ((keys + kSk * tiles - 1) / (kSk * tiles)) < 1024) tiles /= 2;
    const dim3 sg((unsigned)a.nq, (unsigned)((keys + kSk * tiles - 1) / (kSk * tiles)), qg);
    const size_t lds_s = (size_t)((a.hd + 63) / 64 + kSkD) * kStageB;
    moe_status st;
    if ((st = set_lds(attn_scores_qt_kernel, lds_s, "scores LDS attribute"))) return st;
    hipLaunchKernelGGL(attn_scores_qt_kernel, sg, dim3(256), lds_s, s, a, tiles);
    if ((st = check_hip(hipGetLastError(), "scores launch"))) return st;
    // rows a block: 4, fewer where they would not fit two blocks a CU
    int R = kSmRowsMax;
    const size_t row_b = (size_t)sm_row_floats(keys) * 4;
    while (R > 1 && R * row_b > 72 * 1024) R /= 2;
    const size_t lds_m = R * row_b;
    if ((st = set_lds(attn_softmax_rows_kernel, lds_m, "softmax rows LDS attribute"))) return st;
    hipLaunchKernelGGL(attn_softmax_rows_kernel, dim3((unsigned)a.nq, (unsigned)((a.T + R - 1) / R)), dim3(256), lds_m,
                       s, a, R);
    if ((st = check_hip(hipGetLastError(), "softmax rows launch"))) return st;
    hipLaunchKernelGGL(attn_pv_qt_kernel, dim3((unsigned)a.nq, (unsigned)((a.hd + 63) / 64),
                                               (unsigned)((a.T + kPvR - 1) / kPvR)), dim3(256), 0, s, a);
    return check_hip(hipGetLastError(), "softmax/pv launch");
  }
  const int nmax = a.pos0 + a.T;   // positions of the last row
  const size_t hdp = (size_t)((a.hd + 3) & ~3);
  static const bool no_xcd = getenv("MOEHIP_ATTN_NO_XCD") != nullptr;
  AttnArgs ax = a;
  ax.xcd_map = no_xcd ? 0 : 1;
  const dim3 sgrid((unsigned)((nmax + 63) / 64), (unsigned)a.nq, (unsigned)a.T);
  moe_status st;
  if (a.hd <= kRegHd) {
    const size_t lds_s = 10 * hdp * 4;
    hipLaunchKernelGGL(attn_scores_kernel<true>, sgrid, dim3(64), lds_s, s, ax);
  } else {
    const size_t lds_s = (9 * hdp + 64 * (size_t)(a.hd + 4)) * 4;
    if ((st = set_lds(attn_scores_kernel<false>, lds_s, "scores LDS attribute"))) return st;
    hipLaunchKernelGGL(attn_scores_kernel<false>, sgrid, dim3(64), lds_s, s, ax);
  }
  if ((st = check_hip(hipGetLastError(), "scores launch"))) return st;
  const size_t es_f = (size_t)((a.max_seq + 3) & ~3);
  const size_t lds_p = (es_f + kPvDpb * (16384 / kPvDpb + 4)) * 4;
  if ((st = set_lds(attn_softmax_pv_kernel, lds_p, "softmax/pv LDS attribute"))) return st;
  hipLaunchKernelGGL(attn_softmax_pv_kernel, dim3((unsigned)((a.hd + kPvDpb - 1) / kPvDpb), (unsigned)a.nq, (unsigned)a.T),
                     dim3(kPvThreads), lds_p, s, ax);
  return check_hip(hipGetLastError(), "softmax/pv launch");
}

moe_status greedy_vec(const float* v, int n, const float* part, int rows, int32_t* out,
                      int32_t* out_hist, int32_t* hist_pos, hipStream_t s) {
  if (n <= 0) return set_error(MOE_ERR_ARG, "greedy: %d logits", n);
  if (part && rows <= 0) return set_error(MOE_ERR_ARG, "greedy: %d rows per partial", rows);
  hipLaunchKernelGGL(greedy_kernel, dim3(1), dim3(kGreedyThreads), 0, s, v, n, part, rows, out,
                     out_hist, hist_pos);
  return check_hip(hipGetLastError(), "greedy launch");
}

moe_status softmax_vec(float* v, int n, hipStream_t s) {
  hipLaunchKernelGGL(softmax_vec_kernel, dim3(1), dim3(kSmThreads), 0, s, v, n);
  return check_hip(hipGetLastError(), "softmax launch");
}

}  // namespace moe
